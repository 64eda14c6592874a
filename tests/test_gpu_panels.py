"""GPU parity of the prompt panels (csrc/bulk.hip): mi_prefill and mi_teacher run prompts of
9 tokens and more in panels of up to 2048 tokens. Bar: the same bits as one multi-token step
per 7 tokens (tchunk=7, itself bit-identical to single steps and the q8act oracle), in the
predictions, the margins and, through a step's logits, the K/V the panel left.

Lengths sit on the edges of the 32-token tiles, the 64-token GEMM tiles, the panel whose down
matrix is split over workgroups (256), the attention split (1024) and the panel (2048)."""
import sys

import numpy as np
import pytest

import minfer
import oracle_lib as O
from conftest import gguf_tensor, synth_cached, tie_head_gguf

pytestmark = pytest.mark.gpu
# head size 64 with chunks of 8 blocks; head size 128, 7 query heads per kv head, chunks of 4
TINY = dict(n_layer=2, n_embd=256, n_ff=512, n_head=4, n_head_kv=2, n_vocab=4096)
ODD = dict(n_layer=2, n_embd=896, n_ff=1152, n_head=7, n_head_kv=1, n_vocab=4160)
SHAPES = {"hd64": TINY, "hd128-cb4": ODD}


@pytest.fixture(scope="module", autouse=True)
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def bits(x):
    return np.asarray(x, np.float32).view(np.uint32)


@pytest.fixture(scope="module", params=list(SHAPES))
def pair(request):
    """an engine that runs panels and one that runs 7-token steps, the same model"""
    shape = SHAPES[request.param]
    path = synth_cached("panel-" + request.param, shape, 31, qk_bias_std=2.0, norm_offset=1.0)
    a, b = minfer.Engine(path, max_ctx=2112), minfer.Engine(path, max_ctx=2112, tchunk=7)
    yield shape, a, b
    a.close()
    b.close()


@pytest.mark.parametrize("n", [9, 17, 32, 33, 63, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 1151, 2048, 2049])
def test_panel_bit_identical(pair, n):
    shape, a, b = pair
    print("[gpu-panel] n", n, flush=True)
    ids = minfer.prompt_ids(n, n, shape["n_vocab"])
    pa, ma = a.teacher(ids)
    pb, mb = b.teacher(ids)
    assert pa == pb and np.array_equal(bits(ma), bits(mb))
    fa, fb = a.prefill(ids), b.prefill(ids)
    assert fa[0] == fb[0] == pb[-1] and bits(fa[1]) == bits(fb[1])
    _, _, la = a.step(ids[0], n, want_logits=True)
    _, _, lb = b.step(ids[0], n, want_logits=True)
    assert np.array_equal(bits(la), bits(lb))
    a.prefill(ids)
    b.prefill(ids)
    ga, gb = a.generate(1), b.generate(1)       # continues from the panel's prediction
    assert ga[0] == gb[0] and np.array_equal(bits(ga[1]), bits(gb[1]))


def test_panel_infinite_values_stay_with_their_positions(tmpdir_mi):
    """V rows that overflow fp16 at some positions: tokens before them are untouched (a
    masked position adds 0 * V, which must not reach a token that does not see it)"""
    path = synth_cached("panel-hd64", TINY, 31, qk_bias_std=2.0, norm_offset=1.0)
    with open(path, "rb") as f:
        data = bytearray(f.read())
    ty, dims, off = gguf_tensor(path, "blk.1.attn_v.weight")
    assert ty == 2
    nb = dims[0] // 32
    w = np.frombuffer(data, np.uint8, count=nb * 18, offset=off).reshape(nb, 18).copy()
    w[:, :2] = np.full(nb, 900.0, np.float16).view(np.uint8).reshape(nb, 2)
    data[off:off + w.size] = w.tobytes()         # row 0 of V: a sum of order 900 * 4.6 * 16 over 256 terms
    big = tmpdir_mi + "/panel-inf.gguf"
    with open(big, "wb") as f:
        f.write(bytes(data))
    n = 150
    ids = minfer.prompt_ids(3, n, TINY["n_vocab"])
    a, b = minfer.Engine(big, max_ctx=256), minfer.Engine(big, max_ctx=256, tchunk=7)
    pa, ma = a.teacher(ids)
    pb, mb = b.teacher(ids)
    ma, mb = np.float32(ma), np.float32(mb)
    a.close()
    b.close()
    fin = np.isfinite(mb)
    print("[gpu-panel] finite margins", int(fin.sum()), "of", n, flush=True)
    assert 2 <= fin.sum() < n                    # the case has both kinds
    assert np.array_equal(fin, np.isfinite(ma)) and np.array_equal(bits(ma[fin]), bits(mb[fin])) and pa == pb


# the widths of the 0.5B, 1.5B and 3B shapes in two layers, with a small vocabulary
WIDE = {"S05": dict(n_layer=2, n_embd=896, n_ff=4864, n_head=14, n_head_kv=2, n_vocab=4096),
        "S15": dict(n_layer=2, n_embd=1536, n_ff=8960, n_head=12, n_head_kv=2, n_vocab=4096),
        "S3": dict(n_layer=2, n_embd=2048, n_ff=11008, n_head=16, n_head_kv=2, n_vocab=4096)}


@pytest.mark.parametrize("name", list(WIDE))
def test_panel_bit_identical_wide(name):
    """the matrices of the real shapes: down in 19, 35 and 43 chunks (several windows of 8, windows
    that cross a segment), 152 to 344 gate/up row groups (both GEMMs), the norm's second slice"""
    shape = WIDE[name]
    path = synth_cached("panel-wide-" + name, shape, 5, qk_bias_std=2.0, norm_offset=1.0)
    a, b = minfer.Engine(path, max_ctx=640), minfer.Engine(path, max_ctx=640, tchunk=7)
    for n in (9, 64, 65, 128, 256, 257, 320, 513):
        print("[gpu-panel] wide", name, n, flush=True)
        ids = minfer.prompt_ids(n, n, shape["n_vocab"])
        pa, ma = a.teacher(ids)
        pb, mb = b.teacher(ids)
        assert pa == pb and np.array_equal(bits(ma), bits(mb)), n
        fa = a.prefill(ids)
        assert fa[0] == pb[-1] and bits(fa[1]) == bits(mb[-1]), n
        _, _, la = a.step(ids[0], n, want_logits=True)
        _, _, lb = b.step(ids[0], n, want_logits=True)
        assert np.array_equal(bits(la), bits(lb)), n
    a.close()
    b.close()


def test_panel_argmax_ties_first_row(tmpdir_mi):
    """exact logit ties between rows of different row groups: the first row, margin 0, in the
    predictions of every token (teacher) and of the last (prefill)"""
    path = tie_head_gguf(synth_cached("tie-src", TINY, 31), tmpdir_mi + "/panel-tie.gguf", 100, 2000, 7, 3000)
    ids = minfer.prompt_ids(4, 70, TINY["n_vocab"])
    a, b = minfer.Engine(path, max_ctx=128), minfer.Engine(path, max_ctx=128, tchunk=7)
    pa, ma = a.teacher(ids)
    pb, mb = b.teacher(ids)
    first, m = a.prefill(ids)
    a.close()
    b.close()
    assert pa == pb and set(pa) == {100, 7}
    assert not any(ma) and not any(mb)
    assert first == pa[-1] and m == 0.0


def test_panel_denormal_scales(tmpdir_mi):
    """fp16-denormal block scales of weights and activations: their products are exact in the
    panel GEMMs too. Every q4_0 scale is a random denormal and the embedding is small enough for
    the first layer's activation scales to be denormal as well; against 7-token steps and the
    oracle"""
    src = synth_cached("panel-hd64", TINY, 31, qk_bias_std=2.0, norm_offset=1.0)
    with open(src, "rb") as f:
        data = bytearray(f.read())
    rng = np.random.default_rng(8)
    names = ["output.weight"] + ["blk.%d.%s.weight" % (l, t) for l in range(TINY["n_layer"]) for t in (
        "attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")]
    for name in names:
        ty, dims, off = gguf_tensor(src, name)
        assert ty == 2
        nb = dims[0] // 32 * dims[1]
        w = np.frombuffer(data, np.uint8, count=nb * 18, offset=off).reshape(nb, 18).copy()
        w[:, :2] = rng.integers(1, 1024, nb).astype(np.uint16).view(np.uint8).reshape(nb, 2)
        data[off:off + w.size] = w.tobytes()
    ty, dims, off = gguf_tensor(src, "token_embd.weight")
    assert ty == 0
    emb = np.frombuffer(data, np.float32, count=dims[0] * dims[1], offset=off) * np.float32(1e-4)
    data[off:off + 4 * emb.size] = emb.tobytes()
    path = tmpdir_mi + "/panel-denormal.gguf"
    with open(path, "wb") as f:
        f.write(bytes(data))
    ids = minfer.prompt_ids(12, 70, TINY["n_vocab"])
    a, b = minfer.Engine(path, max_ctx=128), minfer.Engine(path, max_ctx=128, tchunk=7)
    p = a.plan
    pa, ma = a.teacher(ids)
    pb, mb = b.teacher(ids)
    _, _, la = a.step(ids[0], 70, want_logits=True)
    _, _, lb = b.step(ids[0], 70, want_logits=True)
    a.close()
    b.close()
    assert pa == pb and np.array_equal(bits(ma), bits(mb)) and np.array_equal(bits(la), bits(lb))
    assert sum(m > 0 for m in ma) > 60            # the products did not vanish
    orc = O.Model(path, O.MODE_Q8ACT, plan=O.Plan.make(p["cb"], p["ks"], p["attn_chunk"], p["kv_f16"]), max_seq=128)
    for i, tok in enumerate(ids):
        t, m = orc.forward(tok, i)
        assert t == pa[i] and bits(m) == bits(ma[i]), i


def test_panel_attention_in_several_launches():
    """contexts whose split records exceed the room kept for them: the attention of a panel goes
    out in two launches (7 heads of 128 over 9 and 10 splits of 1024 positions)"""
    path = synth_cached("panel-hd128-cb4", ODD, 31, qk_bias_std=2.0, norm_offset=1.0)
    n = 9300
    ids = minfer.prompt_ids(n, n, ODD["n_vocab"])
    a, b = minfer.Engine(path, max_ctx=9408), minfer.Engine(path, max_ctx=9408, tchunk=7)
    print("[gpu-panel] long prompt", n, flush=True)
    pa, ma = a.teacher(ids)
    pb, mb = b.teacher(ids)
    assert pa == pb and np.array_equal(bits(ma), bits(mb))
    fa = a.prefill(ids)
    assert fa[0] == pb[-1] and bits(fa[1]) == bits(mb[-1])
    b.prefill(ids)
    _, _, la = a.step(ids[0], n, want_logits=True)
    _, _, lb = b.step(ids[0], n, want_logits=True)
    assert np.array_equal(bits(la), bits(lb))
    a.close()
    b.close()


@pytest.mark.parametrize("opts,limit", [(dict(max_ctx=8), 12), (dict(max_ctx=64, tchunk=7), 12), (dict(max_ctx=64), 12),
                                        (dict(max_ctx=131072, tchunk=7), 300), (dict(max_ctx=131072), 400)],
                         ids=["ctx8", "ctx64-steps", "ctx64", "ctx131072-steps", "ctx131072"])
def test_panel_buffers_fit_the_engine(opts, limit):
    """device memory (MB) of a loaded engine: panel buffers only where panels can run and for no
    more tokens than the context has (2048 tokens' worth of this model's takes 15 MB beside
    the 6 MB of everything else), and bounded split records in a long context (285 MB for 2048
    tokens at once, beside 235 MB of K/V and step records)"""
    import torch
    path = synth_cached("panel-hd64", TINY, 31, qk_bias_std=2.0, norm_offset=1.0)

    def used(**o):
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        e = minfer.Engine(path, **o)
        n = free - torch.cuda.mem_get_info()[0]
        e.close()
        return n / 1e6

    used(max_ctx=64)                             # what the first load of a process adds
    mb = used(**opts)
    print("[gpu-panel] %s: %.1f MB" % (opts, mb), flush=True)
    assert mb <= limit
