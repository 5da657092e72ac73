"""The 32 x 32 tile projections of the batched prefill and of
gsdh_model_matmul at the sizes where their tiling can go wrong, against the
oracle: token counts at the edges of 16-token groups and of the 32- and
64-token tiles (one more and one less), row counts that are not whole row
tiles, columns that end in half a chunk and columns whose chunks do not divide
into the splits, both code formats, kinks and rank-2 terms taken in from
column splits; and that a model takes any number of prompts."""
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


# 8 waves of 32 rows: 256-row tiles that end inside a wave's rows and with
# waves past them, more blocks of operands than CUs, the last group of tokens
# on an XCD of its own round
@pytest.mark.parametrize("M", [65, 144, 257])
@pytest.mark.parametrize("name", ["attn_q", "attn_k", "ffn_gate", "ffn_down"])
def test_matmul_wide_blocks(name, M):
    banner(f"matmul of {M} tokens, {name}, 8 waves")
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
