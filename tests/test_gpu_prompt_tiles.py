"""The 32 x 32 tile projections of the batched prefill and of
gsdh_model_matmul at the sizes where their tiling can go wrong, against the
oracle: token counts at the edges of 16-token groups and of the 32- and
64-token tiles (one more and one less), row counts that are not whole row
tiles, columns that end in half a chunk and columns whose chunks do not divide
into the splits, both code formats, kinks and rank-2 terms taken in from
column splits; the blocks of every width that the choice of tiles gives single
operands, by name; whole layers of the 7B shape; and that a model takes any
number of prompts."""
import ctypes

import numpy as np
import pytest

import oracle as O
from conftest import rel_l2
from gpu_util import D, E, H, banner
from test_gpu_prefill import SLOTS, _kv_close, _pair, _small_model, _spec, bf16, check, layer_shape, run_matmul, turbo_7b  # noqa: F401

pytestmark = pytest.mark.gpu

# hidden 320: chunks of 128, 128 and 64 columns; ffn 832: 6.5 chunks; 5 heads
# of 64: k and v of 320 rows (no whole 128- or 256-row tile)
RAGGED = dict(hidden=320, ffn=832, n_heads=5, n_kv_heads=5, head_dim=64)


# the last position's logits and the cache: fp32 sums of ~22-bit inputs, and
# elements of K / V that round to the other fp16 value (2^-11 of an element)
@pytest.mark.parametrize("n", [1, 2, 16, 17, 31, 32, 33, 63, 64, 65, 129])
@pytest.mark.parametrize("mode,kpr,shape", [("precision", 2, dict()), ("turbo", 1, RAGGED),
                                            ("precision", 0, dict(n_layers=3, hidden=512, ffn=2496, n_heads=8,
                                                                  n_kv_heads=2, head_dim=64))])
def test_prompt_edges(mode, kpr, shape, n):
    banner(f"prompt of {n} tokens, {mode} kinks {kpr} {shape}")
    gpu, ref = _pair(_spec(mode=mode, kinks_per_row=kpr, **shape), max_seq=192)
    toks = np.random.default_rng(n).integers(0, gpu.vocab_size, n).tolist()
    got = gpu.prefill(toks, 0)
    for pos, t in enumerate(toks):
        want = ref.forward_token(t, pos, return_logits=pos == n - 1)
    assert rel_l2(got, want) < 1e-3
    _kv_close(gpu, ref, range(gpu.n_layers), sorted({0, n // 2, n - 1}))
    nxt = int(np.argmax(want))
    assert rel_l2(gpu.forward_token(nxt, n), ref.forward_token(nxt, n)) < 1e-3
    gpu.close()


@pytest.mark.parametrize("M", [1, 31, 33, 65, 113, 127, 129])
@pytest.mark.parametrize("mode,kpr,shape", [("turbo", 1, RAGGED), ("precision", 2, dict(ffn=8256))])
def test_matmul_edges(mode, kpr, shape, M):
    banner(f"matmul of {M} tokens, {mode} kinks {kpr} {shape}")
    src, model = _small_model(_spec(n_layers=1, mode=mode, kinks_per_row=kpr, **shape))
    try:
        for name in ("attn_k", "ffn_up", "ffn_down"):
            key = f"blk.0.{name}.weight"
            t = dict(src.tensors[key])
            for f in ("codes", "scales", "row_ptr", "kink_cols", "kink_deltas") + (("U", "S", "Vt") if t["k_dim"] else ()):
                t[f] = np.ascontiguousarray(src.hex_field(key, f))
            check(model, t, 0, SLOTS[name], M, seed=M + SLOTS[name])
    finally:
        model.close()


# 32-position chunks taken in turn by four pairs of waves: contexts of fewer
# chunks than pairs, one position past and short of a chunk, of a round of
# chunks; 64 query rows of 8, 16, 32 and 64 tokens, and one token more
@pytest.mark.parametrize("p0,M", [(0, 2), (31, 2), (0, 33), (95, 34), (127, 3), (128, 65), (3, 130), (255, 9)])
@pytest.mark.parametrize("nh,nkv,hd", [(8, 1, 128), (4, 4, 64), (4, 2, 128), (16, 4, 64)])
def test_prompt_attention_edges(p0, M, nh, nkv, hd):
    import test_gpu_ops
    from gsdlq import hip
    test_gpu_ops.test_prefill_attention_vs_oracle(hip.lib(), p0, M, nh, nkv, hd, 1, p0 + M + 3)


@pytest.mark.parametrize("mode,shape", [("precision", dict()), ("precision", dict(k_dim=3))])
def test_any_number_of_prompts(mode, shape):
    """Each prompt's head took further publication words of the model until,
    after some two hundred prompts on two layers, none were left."""
    banner(f"300 prompts on one model, {mode} {shape}")
    gpu, ref = _pair(_spec(mode=mode, kinks_per_row=0, **shape), max_seq=16)
    toks = [5, 77, 300]
    for pos, t in enumerate(toks):
        want = ref.forward_token(t, pos, return_logits=pos == 2)
    first = gpu.prefill(toks, 0)
    for _ in range(300):
        got = gpu.prefill(toks, 0)
    assert np.array_equal(first, got)
    assert rel_l2(got, want) < 1e-3
    gpu.close()


# small shapes at batches whose operand pass has more blocks than the chip CUs,
# the last group of tokens on an XCD of its own round; their projections take the
# 16 x 16 tiles (and 4 waves of the 32 x 32 ones at 65 tokens)
@pytest.mark.parametrize("M", [65, 144, 257])
@pytest.mark.parametrize("name", ["attn_q", "attn_k", "ffn_gate", "ffn_down"])
def test_matmul_wide_blocks(name, M):
    banner(f"matmul of {M} tokens, {name}")
    src, model = _small_model(_spec(n_layers=1, mode="turbo", kinks_per_row=1, **RAGGED))
    try:
        key = f"blk.0.{name}.weight"
        t = dict(src.tensors[key])
        for f in ("codes", "scales", "row_ptr", "kink_cols", "kink_deltas"):
            t[f] = np.ascontiguousarray(src.hex_field(key, f))
        check(model, t, 0, SLOTS[name], M, seed=M + SLOTS[name])
    finally:
        model.close()


def _shared(model, names, xb, M, rows):
    lib = model.cl.lib
    dx, ys = D(xb), [E(M * r * 4) for r in rows]
    slots = (ctypes.c_int * len(names))(*[SLOTS[n] for n in names])
    lib.gsdh_model_matmul_shared(model._m, 0, slots, len(names), dx.ptr, M,
                                 (ctypes.c_void_p * len(names))(*[y.ptr.value for y in ys]))
    lib.gsdh_stream_sync(lib.gsdh_model_stream(model._m))
    return [H(y, np.float32, M * r).reshape(M, r) for y, r in zip(ys, rows)]


# sets whose partial sums fit the workspace together, and sets that take a
# launch for each tensor or two: any tensors of equal columns share a call
@pytest.mark.parametrize("names,M", [(("ffn_down",) * 3, 512), (("ffn_gate", "attn_q", "ffn_up"), 128),
                                     (("ffn_gate",) * 3, 128), (("attn_output", "attn_q", "attn_q"), 64)])
def test_matmul_any_set_equals_separate_calls(turbo_7b, names, M):  # noqa: F811
    banner(f"shared-input matmul {names} M={M}")
    _, model = turbo_7b
    rows = [layer_shape(n)[0] for n in names]
    xb, _ = bf16(np.random.default_rng(M).standard_normal((M, layer_shape(names[0])[1])).astype(np.float32))
    want = {n: run_matmul(model, 0, SLOTS[n], xb, M, r) for n, r in zip(names, rows)}
    for n, got in zip(names, _shared(model, names, xb, M, rows)):
        assert np.array_equal(got, want[n]), n


def test_model_memory(turbo_7b):  # noqa: F811
    """A model's memory beyond its tensors, embedding and cache: the partial
    sums of the largest set of tensors that share an input (33.5 MB, down at 512
    tokens), and no copy of the inputs for kink terms that it does not have."""
    _, model = turbo_7b
    packed = sum(r * c // 2 + r * c // 32 for r, c in [layer_shape(n) for n in SLOTS] + [(32768, 4096)])
    slabs = 4096 * 14336 // 2 + 4096 * 14336 // 32       # down again, for the fused launch
    embedding, cache = 2 * 32768 * 4096, 4 * 640 * 1024
    rest = model.cl.allocated_bytes - packed - slabs - embedding - cache
    tokens = 512
    prompt = 4 * tokens * (2 * 4096 + 2 * 1024 + 4096 + 2 * 14336) + 8 * tokens * 14336
    operands, parts = 4 * tokens * 14336, 4 * 4 * tokens * 4096
    print(f"[gpu-test] beyond tensors, embedding and cache: {rest / 1e6:.1f} MB "
          f"({(rest - prompt - operands - parts) / 1e6:.1f} above the prompt's rows, the operands and one set's sums)", flush=True)
    assert rest - prompt - operands - parts < 20e6       # (the prompts' own partial sums, decode's hand-off words)


def _tile(model, M, t):
    w, n = ctypes.c_int(), ctypes.c_int()
    r = t["radius"]
    model.cl.lib.gsdh_matmul_tile(M, t["rows"], t["cols"], 3 * r * r + 3 * r + 1, ctypes.byref(w), ctypes.byref(n))
    return w.value, n.value


def _tensor(src, key):
    t = dict(src.tensors[key])
    for f in ("codes", "scales", "row_ptr", "kink_cols", "kink_deltas") + (("U", "S", "Vt") if t["k_dim"] else ()):
        t[f] = np.ascontiguousarray(src.hex_field(key, f))
    return t


def _some(M):
    return sorted({0, 15, 16, 31, 32, 63, 64, M // 2, M - 17, M - 1} & set(range(M)))


# every block of single operands (waves, tokens) that the choice gives the 7B
# shapes, split and unsplit, at token counts that end inside a tile
@pytest.mark.parametrize("name,M,tile", [
    ("ffn_down", 9, (4, 32)), ("ffn_down", 50, (4, 64)), ("ffn_down", 65, (4, 128)), ("ffn_down", 129, (8, 64)),
    ("ffn_down", 300, (8, 64)), ("ffn_down", 447, (8, 64)), ("ffn_down", 511, (4, 128)), ("ffn_gate", 257, (8, 64)),
    ("ffn_gate", 448, (8, 64)), ("ffn_gate", 509, (4, 128)), ("attn_k", 33, (4, 64)), ("attn_q", 513 - 1, (0, 0))])
def test_matmul_blocks_7b(turbo_7b, name, M, tile):  # noqa: F811
    bank, model = turbo_7b
    t = bank.packed[(0, name)]
    banner(f"matmul 7B turbo {name} M={M}, {tile[0]} waves over {tile[1]} tokens")
    assert _tile(model, M, t) == tile
    check(model, t, 0, SLOTS[name], M, seed=M + SLOTS[name], tokens=_some(M))


# 8 waves over tall tensors whose last 256-row tile ends inside a wave's rows
# (14308 = 55 x 256 + 7 x 32 + 4) and before its last waves (14404: + 2 x 32 + 4),
# both code formats, with kinks and ranks 0 to 2
@pytest.mark.parametrize("mode,k_dim,vocab", [("turbo", 0, 14308), ("precision", 2, 14404), ("precision", 1, 14308)])
@pytest.mark.parametrize("M", [257, 320, 385])
def test_matmul_wide_blocks_tall(mode, k_dim, vocab, M):
    banner(f"matmul of {M} tokens, head of {vocab} rows, {mode} rank {k_dim}, 8 waves")
    src, model = _small_model(_spec(n_layers=1, mode=mode, k_dim=k_dim, kinks_per_row=1, vocab=vocab))
    try:
        t = _tensor(src, "output.weight")
        assert _tile(model, M, t) == (8, 64)
        check(model, t, 0, 7, M, seed=M, tokens=_some(M))
    finally:
        model.close()


# 8 waves over split columns with rank and kink terms, 7-bit codes (3072 x 14336)
def test_matmul_wide_blocks_split():
    banner("matmul of 129 tokens, 3072 x 14336, precision with kinks, 8 waves, split")
    src, model = _small_model(_spec(n_layers=1, mode="precision", kinks_per_row=2, hidden=3072, ffn=14336, n_heads=24,
                                    n_kv_heads=6, head_dim=128))
    try:
        t = _tensor(src, "blk.0.ffn_down.weight")
        assert _tile(model, 129, t) == (8, 64)
        check(model, t, 0, SLOTS["ffn_down"], 129, seed=5, tokens=_some(129))
    finally:
        model.close()


class _MixedRanks:
    """A packed model whose tensors have ranks of their own (0, 1 or 2)."""

    def __init__(self, ranks, **kw):
        from gsdlq import synth
        spec = _spec(mode="precision", **kw)
        of = [synth.SynthSource(_spec(mode="precision", k_dim=k, **kw)) for k in range(3)]
        self.by_name = {n: of[ranks.get(n.split(".")[-2], 2)] for n in synth.tensor_shapes(spec)}
        self.config, self.header = of[0].config, {"avg_bpw": None}
        self.tensors = {**of[0].tensors, **{n: s.tensors[n] for n, s in self.by_name.items()}}
        self.dense = of[0].dense

    def hex_field(self, name, field):
        return self.by_name[name].hex_field(name, field)

    def close(self):
        pass


RANKS = [dict.fromkeys(SLOTS, 1), dict(attn_q=2, attn_k=0, attn_v=1, attn_output=0, ffn_gate=1, ffn_up=2, ffn_down=1)]


@pytest.mark.parametrize("ranks", RANKS, ids=["rank1", "mixed"])
@pytest.mark.parametrize("n", [3, 70])
def test_prompt_ranks(ranks, n):
    import run_gpu_native_chat as chat
    banner(f"prompt of {n} tokens, ranks {ranks}")
    src = _MixedRanks(ranks, kinks_per_row=1)
    gpu = chat.GPUMistralV2Model(src, max_seq_len=96, verbose=False)
    ref = O.OracleModel(src, kind="port", max_seq_len=96)
    toks = np.random.default_rng(n).integers(0, gpu.vocab_size, n).tolist()
    got = gpu.prefill(toks, 0)
    for pos, t in enumerate(toks):
        want = ref.forward_token(t, pos, return_logits=pos == n - 1)
    assert rel_l2(got, want) < 1e-3
    _kv_close(gpu, ref, range(gpu.n_layers), sorted({0, n // 2, n - 1}))
    gpu.close()


@pytest.mark.parametrize("ranks", RANKS, ids=["rank1", "mixed"])
@pytest.mark.parametrize("names", [("attn_q", "attn_k", "attn_v"), ("ffn_gate", "ffn_up"), ("ffn_down",)])
def test_matmul_ranks(ranks, names, M=21):
    import run_gpu_native_chat as chat
    banner(f"matmul of {M} tokens, {names}, ranks {ranks}")
    src = _MixedRanks(ranks, n_layers=1, kinks_per_row=1)
    model = chat.GPUMistralV2Model(src, max_seq_len=64, verbose=False)
    ts = [_tensor(src, f"blk.0.{n}.weight") for n in names]
    assert all(_tile(model, M, t)[0] for t in ts)
    xb, xf = bf16(np.random.default_rng(3).standard_normal((M, ts[0]["cols"])).astype(np.float32))
    for t, got in zip(ts, _shared(model, names, xb, M, [t["rows"] for t in ts])):
        for m in range(M):
            assert rel_l2(got[m], O.hex2d_matvec(xf[m], t)) < 1e-3, m
    model.close()


# X or Y off the 16 bytes that the one-pass operands and the 32 x 32 tiles need,
# and rows of X too long for that pass: the older launches serve them
@pytest.mark.parametrize("x_off,y_off,ffn", [(2, 0, 512), (8, 0, 512), (0, 4, 512), (0, 8, 512), (2, 12, 512), (0, 0, 16448)])
@pytest.mark.parametrize("name", ["attn_q", "ffn_down"])
def test_matmul_other_routes(x_off, y_off, ffn, name, M=40):
    banner(f"matmul of {M} tokens, {name}, X off by {x_off}, Y off by {y_off} bytes, ffn {ffn}")
    src, model = _small_model(_spec(n_layers=1, mode="precision", kinks_per_row=1, ffn=ffn))
    lib, t = model.cl.lib, _tensor(src, f"blk.0.{name}.weight")
    rows, cols = t["rows"], t["cols"]
    xb, xf = bf16(np.random.default_rng(M).standard_normal((M, cols)).astype(np.float32))
    dx, dy = D(np.concatenate([np.zeros(x_off // 2, np.uint16), xb.reshape(-1)])), E(M * rows * 4 + 16)
    lib.gsdh_model_matmul(model._m, 0, SLOTS[name], dx.ptr.value + x_off, M, dy.ptr.value + y_off)
    lib.gsdh_stream_sync(lib.gsdh_model_stream(model._m))
    out = H(dy, np.float32)
    got = out[y_off // 4:][:M * rows].reshape(M, rows)
    assert not out[:y_off // 4].any() and not out[y_off // 4 + M * rows:].any()
    for m in range(M):
        assert rel_l2(got[m], O.hex2d_matvec(xf[m], t)) < 1e-3, m
    model.close()


# A prompt's whole layers at the 7B widths (the last layer forms K and V alone
# for all but one token, so one layer shows none of the rest): 513 tokens, a
# chunk of 512 (8 waves over 64 tokens; 784- and 896-block grids, 14336-column
# operand rows) and one of a single token; then 64 behind them
@pytest.mark.parametrize("mode,kpr", [("turbo", 0), ("precision", 1)])
def test_prompt_7b_layers(mode, kpr):
    banner(f"two layers of the 7B shape, {mode} kinks {kpr}: prompts of 513, then 64")
    gpu, ref = _pair(_spec(mode=mode, kinks_per_row=kpr, hidden=4096, ffn=14336, n_heads=32, n_kv_heads=8, head_dim=128),
                     max_seq=640)
    toks = np.random.default_rng(8).integers(0, gpu.vocab_size, 577).tolist()
    for a, b in ((0, 513), (513, 577)):
        got = gpu.prefill(toks[a:b], a)
        for pos in range(a, b):
            want = ref.forward_token(toks[pos], pos, return_logits=pos == b - 1)
        e = rel_l2(got, want)
        print(f"[prefill-parity] 7B {mode}, two layers, positions {a}..{b - 1}: logits rel L2 {e:.2e}", flush=True)
        assert e < 1e-3
        _kv_close(gpu, ref, [0, 1], [a, (a + b) // 2, b - 2, b - 1])
    gpu.close()


# head dim 128, four query heads per KV head and an ffn that ends in half a
# chunk, with a layer before the last
def test_prompt_ragged_two_layers():
    n = 130
    gpu, ref = _pair(_spec(mode="turbo", kinks_per_row=1, hidden=512, ffn=1344, n_heads=8, n_kv_heads=2, head_dim=128,
                           vocab=1000))
    banner(f"prompt of {n} tokens, hd 128, ragged ffn, two layers")
    toks = np.random.default_rng(n).integers(0, gpu.vocab_size, n).tolist()
    got = gpu.prefill(toks, 0)
    for pos, t in enumerate(toks):
        want = ref.forward_token(t, pos, return_logits=pos == n - 1)
    assert rel_l2(got, want) < 1e-3
    _kv_close(gpu, ref, [0, 1], [0, 64, n - 1])
    gpu.close()


def test_prompt_without_logits_leaves_the_state():
    """A prompt without logits leaves the last token's state for the head
    alone (gsdh_model_run_linear) and for gsdh_model_vector."""
    from gsdlq import hip
    banner("prompt without logits, then the head")
    gpu, _ = _pair(_spec())
    toks = np.random.default_rng(2).integers(0, gpu.vocab_size, 37).tolist()
    want = gpu.prefill(toks, 0)
    other = gpu.prefill(toks[::-1], 0)
    gpu.prefill(toks, 0, return_logits=False)
    lib, got = gpu.cl.lib, np.empty(gpu.vocab_size, np.float32)
    lib.gsdh_model_run_linear(gpu._m, 0, 16)
    lib.gsdh_model_vector(gpu._m, hip.VECTORS["logits"], 0, hip.ptr(got), got.nbytes)
    assert np.array_equal(got, want) and not np.array_equal(got, other)
    gpu.close()
