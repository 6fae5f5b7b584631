"""Exact attention of a prompt chunk on the matrix cores: every token's output
reaches the next layer's K / V rows, so those rows and the last logits equal
the oracle decoder's bit for bit."""
import numpy as np
import pytest

from conftest import tiny_llama
from oracle import oracle as ref

pytestmark = pytest.mark.gpu


def run_both(m, chunks, max_len):
    from gopherllm_amd.decoder import LlamaDecoder
    gpu, cpu = LlamaDecoder.from_host_model(m, max_len), ref.Llama(m, max_len)
    pos = 0
    for c in chunks:
        _, gl = gpu.prefill(c, start_pos=pos, want_logits=True)
        _, cl = cpu.prefill(c, start_pos=pos)
        pos += len(c)
    layers = m["config"]["n_layers"]
    kv = gpu.kv_cache()
    rows = [(kv.read(l, 0, pos), (cpu.kcache(l, max_len)[:pos], cpu.vcache(l, max_len)[:pos]))
            for l in range(layers)]
    return (gl, cl), rows


# query heads per kv head 1, 3, 4 and 8 (row tiles that split a token's heads),
# both head sizes; a tile's last rows past the chunk, spans just short of,
# on and past 16, 64 and 128 positions
@pytest.mark.parametrize("heads,n_kv,hd,start,p", [
    (8, 2, 128, 0, 16), (4, 4, 128, 5, 17), (8, 1, 128, 63, 33), (12, 4, 64, 130, 19), (8, 2, 64, 1, 64),
    (4, 1, 128, 0, 130), (8, 2, 128, 127, 15), (12, 4, 64, 126, 3), (8, 8, 64, 40, 24)])
def test_prompt_attention_bit_exact(hip, heads, n_kv, hd, start, p):
    m = tiny_llama(seed=70 + p, n_layers=2, dim=512, hidden=512, n_heads=heads, n_kv_heads=n_kv, head_dim=hd,
                   vocab=600)
    toks = np.random.default_rng(71 + p).integers(0, 600, start + p)
    chunks = [toks[:start], toks[start:]] if start else [toks]
    print(f"{heads}/{n_kv} heads of {hd}, {p} tokens at {start}", flush=True)
    (gl, cl), rows = run_both(m, chunks, start + p + 3)
    assert np.array_equal(gl.view(np.uint32), np.asarray(cl, np.float32).view(np.uint32))
    for l, ((gk, gv), (ck, cv)) in enumerate(rows):
        assert np.array_equal(gk, ck) and np.array_equal(gv, cv), l


def test_infinite_value_row_reaches_later_tokens_only(hip):
    """One token's V row overflows f16 in one element.  The tokens before it,
    in its own 16-row tile too, have weight 0 for that row, and 0 * inf must
    not reach them."""
    m = tiny_llama(seed=90, n_layers=2, dim=512, hidden=512, n_heads=4, n_kv_heads=1, head_dim=128, vocab=600)
    rng = np.random.default_rng(91)
    emb = rng.standard_normal((600, 512), dtype=np.float32) * np.float32(0.02)
    emb[599] = 0.0
    emb[599, 0] = 1.0  # normalised: sqrt(512) in element 0
    wv = rng.standard_normal((128, 512), dtype=np.float32) * np.float32(0.02)
    wv[3, 0] = 5000.0
    m["tok_embd"] = ref.quantize_rows(m["config"]["emb_type"], emb)
    m["wv"][0] = ref.quantize_rows(m["config"]["layer_type"], wv)
    toks = rng.integers(0, 599, 70)
    first = 38
    toks[first] = 599
    _, rows = run_both(m, [toks], 80)
    (_, gv0), (_, cv0) = rows[0]
    assert np.array_equal(gv0, cv0) and np.isinf(gv0[first].view(np.float16)).any()
    (gk, gv), (ck, cv) = rows[1]
    assert np.array_equal(gk[:first], ck[:first]) and np.array_equal(gv[:first], cv[:first])
    assert np.isfinite(gk[:first].view(np.float16)).all()
    for a, b in ((gk, ck), (gv, cv)):
        assert np.array_equal(np.isnan(a.view(np.float16)), np.isnan(b.view(np.float16)))


def test_infinite_key_row_bit_exact(hip):
    """One token's K row overflows f16 in one element: the query rows that reach
    it have an infinite score there, of either sign (NaN outputs, or a weight
    of 0), the tokens before it in its own tile none."""
    m = tiny_llama(seed=92, n_layers=2, dim=512, hidden=512, n_heads=4, n_kv_heads=1, head_dim=128, vocab=600)
    rng = np.random.default_rng(93)
    emb = rng.standard_normal((600, 512), dtype=np.float32) * np.float32(0.02)
    emb[599] = 0.0
    emb[599, 0] = 1.0
    wk = rng.standard_normal((128, 512), dtype=np.float32) * np.float32(0.02)
    wk[127, 0] = 3500.0  # rotated slowest, so that element 63 or 127 alone overflows
    m["tok_embd"] = ref.quantize_rows(m["config"]["emb_type"], emb)
    m["wk"][0] = ref.quantize_rows(m["config"]["layer_type"], wk)
    toks = rng.integers(0, 599, 70)
    first = 38
    toks[first] = 599
    _, rows = run_both(m, [toks], 80)
    (gk0, _), (ck0, _) = rows[0]
    assert np.array_equal(gk0, ck0) and np.isinf(gk0[first].view(np.float16)).any()
    (gk, gv), (ck, cv) = rows[1]
    assert np.isfinite(gk[:first].view(np.float16)).all()
    for a, b in ((gk, ck), (gv, cv)):
        nan = np.isnan(b.view(np.float16))
        assert np.array_equal(np.isnan(a.view(np.float16)), nan)
        assert np.array_equal(a[~nan], b[~nan])


# a second pass over the rows' chunk maxima (past 2560 positions), fewer than 16
# tokens whose spans pass what the one-token kernels keep in LDS (6144), and a
# head size that keeps the three general kernels
@pytest.mark.parametrize("heads,n_kv,hd,start,p", [(4, 1, 128, 2700, 40), (8, 1, 128, 5200, 17), (4, 1, 128, 6139, 9),
                                                   (8, 2, 96, 0, 40), (8, 2, 96, 70, 5)])
def test_prompt_attention_over_a_filled_cache(hip, heads, n_kv, hd, start, p):
    from gopherllm_amd.decoder import LlamaDecoder
    m = tiny_llama(seed=94, n_layers=2, dim=256, hidden=1024, n_heads=heads, n_kv_heads=n_kv, head_dim=hd, vocab=600)
    max_len, kvd = start + p + 5, n_kv * hd
    rng = np.random.default_rng(95 + start)
    gpu, cpu = LlamaDecoder.from_host_model(m, max_len), ref.Llama(m, max_len)
    kv = gpu.kv_cache()
    for l in range(2 if start else 0):
        k, v = (rng.standard_normal((start, kvd), dtype=np.float32) for _ in range(2))
        for pos in range(start):
            kv.store_kv(l, pos, k[pos], v[pos])
        cpu.set_kv(l, 0, ref.f32_to_f16(k), ref.f32_to_f16(v))
    toks = rng.integers(0, 600, p)
    print(f"{heads}/{n_kv} heads of {hd}, {p} tokens at {start}", flush=True)
    gt, gl = gpu.prefill(toks, start_pos=start, want_logits=True)
    ct, cl = cpu.prefill(toks, start_pos=start)
    assert gt == ct
    assert np.array_equal(gl.view(np.uint32), np.asarray(cl, np.float32).view(np.uint32))
    # the second layer's rows hold every token's output of the first
    gk, gv = kv.read(1, start, p)
    assert np.array_equal(gk, cpu.kcache(1, max_len)[start:start + p])
    assert np.array_equal(gv, cpu.vcache(1, max_len)[start:start + p])
