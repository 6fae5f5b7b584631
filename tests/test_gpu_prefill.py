"""Batched prefill products: Q4_K, Q6_K and Q8_0 on the matrix
cores.

matvecBatchQ8 (kernels_amd64.go:470-581) evaluates q4kDotQ8KRow once per
(row, token), so the batched result must equal the per-token row kernel bit
for bit: checked against the amd64-order oracle on small shapes (ragged row
and token tiles, degenerate activation blocks) and, at the configs[2] sizes,
against the oracle on sampled tokens plus the GPU's own batch-1 path on every
token (the reference's batched == per-token invariant, forward_batch_test.go).
"""
import numpy as np
import pytest

from conftest import extreme_row, normal, quant_matrix, random_rows
from oracle import oracle as ref

pytestmark = pytest.mark.gpu


def bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def amd64(data, xs, rows, cols, qtype=ref.Q4_K):
    want = ref.matvec_batch_fast(qtype, data, xs, rows, cols)
    if want is None:
        want = ref.matvec_batch(qtype, data, xs, rows, cols)
    return want.reshape(xs.shape[0], rows)


def assert_bits(got, want, what):
    bad = np.argwhere(bits(got) != bits(want))
    assert bad.size == 0, f"{what}: {len(bad)} values differ, first (token, row) {bad[:4].tolist()}: " \
        f"{got[tuple(bad[0])]} vs {want[tuple(bad[0])]}"


def matvec_group(hip, ws, xs):
    """One call for weights that share their input."""
    import torch
    x = torch.from_numpy(xs).cuda()
    outs = [torch.full((len(xs), w.rows), -1.0, device="cuda") for w in ws]
    hip.matvec_multi_dev(ws, x, outs)
    torch.cuda.synchronize()
    return [o.cpu().numpy() for o in outs]


@pytest.mark.parametrize("rows,cols,p", [(300, 1024, 16), (300, 1024, 33), (64, 256, 100),
                                         (1000, 4096, 64), (70, 14336, 40)])
def test_prefill_bit_exact_small(hip, rows, cols, p):
    data, _ = quant_matrix(ref.Q4_K, rows, cols, 500 + p + rows)
    w = hip.Weight.from_host(data, ref.Q4_K, rows, cols)
    xs = normal(501 + p, (p, cols))
    print(f"prefill {rows}x{cols} p={p}", flush=True)
    got = w.matvec_batch(xs)
    assert_bits(got, amd64(data, xs, rows, cols), "vs amd64 oracle")


@pytest.mark.parametrize("rows,cols,p", [(1, 768, 17), (65, 256, 65), (64, 512, 128), (130, 1280, 129),
                                         (63, 768, 64)])
def test_prefill_tile_edges(hip, rows, cols, p):
    """One row or token past a 64 x 64 tile, one to five blocks (the block
    loop's two halves), the last wave's rows and tokens past the end."""
    data, _ = quant_matrix(ref.Q4_K, rows, cols, 900 + rows)
    w = hip.Weight.from_host(data, ref.Q4_K, rows, cols)
    xs = normal(901 + p, (p, cols))
    assert_bits(w.matvec_batch(xs), amd64(data, xs, rows, cols), f"{rows}x{cols} p={p}")


@pytest.mark.parametrize("rows,cols,p", [(1, 2048, 17), (65, 2048, 65), (64, 4096, 128), (130, 2048, 129)])
def test_prefill_q6k_tile_edges(hip, rows, cols, p):
    data, _ = quant_matrix(ref.Q6_K, rows, cols, 910 + rows)
    w = hip.Weight.from_host(data, ref.Q6_K, rows, cols)
    xs = normal(911 + p, (p, cols))
    assert_bits(w.matvec_batch(xs), amd64(data, xs, rows, cols, ref.Q6_K), f"{rows}x{cols} p={p}")


@pytest.mark.parametrize("rows,cols,p", [(1, 256, 17), (65, 768, 65), (64, 512, 128), (130, 1280, 129)])
def test_prefill_q8_0_tile_edges(hip, rows, cols, p):
    data, _ = quant_matrix(ref.Q8_0, rows, cols, 920 + rows)
    w = hip.Weight.from_host(data, ref.Q8_0, rows, cols)
    xs = normal(921 + p, (p, cols))
    assert_bits(w.matvec_batch(xs), amd64(data, xs, rows, cols, ref.Q8_0), f"{rows}x{cols} p={p}")


@pytest.mark.parametrize("rows,cols,p", [(1, 256, 17), (65, 768, 65), (64, 512, 128), (130, 4096, 129)])
def test_prefill_q5k_tile_edges(hip, rows, cols, p):
    """Q5_K on the Q4_K kernel's tiles; the last row has every code, scale and
    min at its maximum (sc * code = 63 * 31, the largest f16 operand)."""
    data = random_rows(ref.Q5_K, rows, cols, 940 + rows)
    data[-(cols // 256) * 176:] = extreme_row(ref.Q5_K, cols)
    w = hip.Weight.from_host(data, ref.Q5_K, rows, cols)
    xs = normal(941 + p, (p, cols))
    xs[p - 1] = 127.0
    assert_bits(w.matvec_batch(xs), amd64(data, xs, rows, cols, ref.Q5_K), f"{rows}x{cols} p={p}")


@pytest.mark.parametrize("rows,cols,p", [(1, 256, 17), (65, 768, 65), (64, 512, 128), (130, 4096, 129)])
def test_prefill_q4_0_tile_edges(hip, rows, cols, p):
    """Every code at its maximum in the last row, and a token of zeros."""
    data = random_rows(ref.Q4_0, rows, cols, 950 + rows)
    data[-(cols // 32) * 18:] = extreme_row(ref.Q4_0, cols)
    w = hip.Weight.from_host(data, ref.Q4_0, rows, cols)
    xs = normal(951 + p, (p, cols))
    xs[p // 2] = 0.0
    xs[p - 1] = 127.0
    assert_bits(w.matvec_batch(xs), amd64(data, xs, rows, cols, ref.Q4_0), f"{rows}x{cols} p={p}")


@pytest.mark.parametrize("qtype", [ref.Q4_K, ref.Q5_K, ref.Q6_K, ref.Q8_0, ref.Q4_0])
@pytest.mark.parametrize("p", [32, 33, 96, 97])
def test_prefill_half_token_tiles(hip, qtype, p):
    """32 tokens run two of the 64-token tile's four token tiles, 33 all; the
    same counts behind a full tile."""
    rows, cols = 70, 2048
    data = (quant_matrix(qtype, rows, cols, 960 + p)[0] if qtype in (ref.Q4_K, ref.Q6_K, ref.Q8_0)
            else random_rows(qtype, rows, cols, 960 + p))
    w = hip.Weight.from_host(data, qtype, rows, cols)
    xs = normal(961 + p, (p, cols))
    assert_bits(w.matvec_batch(xs), amd64(data, xs, rows, cols, qtype), f"type {qtype} p={p}")


@pytest.mark.parametrize("qtype", [ref.Q4_K, ref.Q6_K])
@pytest.mark.parametrize("rows,cols,p", [(1, 6144, 2), (17, 2048, 5), (40, 6144, 8), (33, 4096, 9), (16, 2048, 16),
                                         (8200, 2048, 7), (8200, 2048, 13), (20, 8192, 4)])
def test_small_batch_edges(hip, qtype, rows, cols, p):
    """One to three row tiles with a short last one, both token widths with and
    without padding, both splits of the lane pairs, block counts that end a
    turn of the ring and, for Q4_K, ones that do not."""
    if qtype == ref.Q4_K:
        cols += 256
    data, _ = quant_matrix(qtype, rows, cols, 930 + rows)
    w = hip.Weight.from_host(data, qtype, rows, cols)
    xs = normal(931 + p, (p, cols))
    xs[p // 2, :256] = 0.0
    assert_bits(w.matvec_batch(xs), amd64(data, xs, rows, cols, qtype), f"{rows}x{cols} p={p}")


@pytest.mark.parametrize("qtype", [ref.Q4_K, ref.Q6_K])
@pytest.mark.parametrize("rows,cols,p", [((33, 16, 1), 6144, 5), ((4100, 1040), 2048, 8), ((4097, 1024, 3100), 2048, 6),
                                         ((17, 40, 48), 6144, 13), ((16, 500), 8192, 4)])
def test_small_batch_groups(hip, qtype, rows, cols, p):
    """Two and three weights in one grid: short last row tiles, a weight of one
    row, enough workgroups for either split of the lane pairs."""
    xs = normal(991 + p, (p, cols))
    data = [quant_matrix(qtype, r, cols, 990 + i)[0] for i, r in enumerate(rows)]
    got = matvec_group(hip, [hip.Weight.from_host(d, qtype, r, cols) for d, r in zip(data, rows)], xs)
    for i, (d, r) in enumerate(zip(data, rows)):
        assert_bits(got[i], amd64(d, xs, r, cols, qtype), f"weight {i} of {rows} x {cols} p={p}")


@pytest.mark.parametrize("rows,cols,p", [(10816, 512, 12), (10817, 768, 9), (10830, 2304, 15), (20480, 256, 8),
                                         (20479, 256, 8), (24576, 1024, 6), (24576, 1024, 7), (4100, 8192, 2),
                                         (4090, 8192, 2), (6144, 8192, 3), (8192, 2048, 16)])
def test_small_batch_routes(hip, rows, cols, p):
    """Both sides of the lines between the small-batch kernel, the row kernels
    and the 64 x 16 tiles (one block or an odd count, short last row tiles,
    fewer than 16 tokens)."""
    data = np.tile(quant_matrix(ref.Q4_K, 50, cols, 995)[0], -(-rows // 50))[:rows * (cols // 256) * 144]
    w = hip.Weight.from_host(data, ref.Q4_K, rows, cols)
    xs = normal(996 + p, (p, cols))
    assert_bits(w.matvec_batch(xs), amd64(data, xs, rows, cols), f"{rows}x{cols} p={p}")


@pytest.mark.parametrize("p", [5, 8, 11, 16])
def test_small_batch_wide_rows(hip, p):
    """257 blocks and one row past the row tiles, both token widths."""
    rows, cols = 65, 65792
    data, _ = quant_matrix(ref.Q4_K, rows, cols, 980)
    w = hip.Weight.from_host(data, ref.Q4_K, rows, cols)
    xs = normal(981 + p, (p, cols))
    assert_bits(w.matvec_batch(xs), amd64(data, xs, rows, cols), f"{rows}x{cols} p={p}")


@pytest.mark.parametrize("p", [6, 9])
def test_small_batch_few_rows_past_4_gib(hip, p):
    """8192 rows of 512 KB: a weight of 4 GiB with too few rows for the 64 x 16
    tiles to cover the GPU still runs on them, and on the row kernel below 8
    tokens."""
    import torch
    rows, cols = 32, 256 * 3641
    data, _ = quant_matrix(ref.Q4_K, rows, cols, 982)
    times = 8192 // rows
    raw = torch.from_numpy(data).cuda().repeat(times)
    assert raw.numel() > 1 << 32
    w = hip.Weight.from_device(raw, ref.Q4_K, 8192, cols)
    del raw
    xs = normal(983, (p, cols))
    out = torch.full((p, 8192), -1.0, device="cuda")
    print(f"8192 x {cols}, {p} tokens", flush=True)
    w.matvec_dev(torch.from_numpy(xs).cuda(), out)
    torch.cuda.synchronize()
    want = torch.from_numpy(amd64(data, xs, rows, cols)).cuda()
    assert (out.view(torch.int32).view(p, times, rows) == want.view(torch.int32)[:, None]).all()
    del w
    torch.cuda.empty_cache()


@pytest.mark.parametrize("qtype,p", [(ref.Q8_0, 17), (ref.Q6_K, 17), (ref.Q5_K, 17), (ref.Q4_0, 17), (ref.Q4_K, 9)])
def test_group_with_a_weight_past_4_gib(hip, qtype, p):
    """The kernels with 32-bit offsets look at every weight of a group: 64 rows
    beside the same rows repeated past 4 GiB."""
    import torch
    cols = 4096
    data = (quant_matrix(qtype, 64, cols, 997)[0] if qtype in (ref.Q4_K, ref.Q6_K, ref.Q8_0)
            else random_rows(qtype, 64, cols, 997))
    times = (1 << 32) // len(data) + 1
    raw = torch.from_numpy(data).cuda().repeat(times)
    assert raw.numel() > 1 << 32
    ws = [hip.Weight.from_host(data, qtype, 64, cols), hip.Weight.from_device(raw, qtype, 64 * times, cols)]
    del raw
    xs = normal(998, (p, cols))
    x = torch.from_numpy(xs).cuda()
    outs = [torch.full((p, w.rows), -1.0, device="cuda") for w in ws]
    print(f"type {qtype}, weights of 64 and {64 * times} rows", flush=True)
    hip.matvec_multi_dev(ws, x, outs)
    torch.cuda.synchronize()
    want = torch.from_numpy(amd64(data, xs, 64, cols, qtype)).cuda()
    assert torch.equal(outs[0].view(torch.int32), want.view(torch.int32))
    assert (outs[1].view(torch.int32).view(p, times, 64) == want.view(torch.int32)[:, None]).all()
    del ws, outs
    torch.cuda.empty_cache()


def test_prefill_degenerate_blocks(hip):
    """All-zero tokens, zero 256-blocks inside a token, a lone large value and
    NaN-free extremes (q8kQuantize's scale-0 blocks, quant_q8k_portable.go:36-62)."""
    rows, cols, p = 130, 1024, 20
    data, _ = quant_matrix(ref.Q4_K, rows, cols, 77)
    w = hip.Weight.from_host(data, ref.Q4_K, rows, cols)
    xs = normal(78, (p, cols))
    xs[0] = 0.0
    xs[3, 256:512] = 0.0
    xs[5, :] = 0.0
    xs[5, 700] = -3.5
    xs[7] *= 1e4
    xs[9] = np.float32(1e-30)
    got = w.matvec_batch(xs)
    assert_bits(got, amd64(data, xs, rows, cols), "degenerate activations")


@pytest.mark.parametrize("qtype", [ref.Q4_K, ref.Q5_K, ref.Q6_K, ref.Q8_0, ref.Q4_0])
@pytest.mark.parametrize("p", [3, 8, 16, 17, 40])
def test_tiny_activations(hip, qtype, p):
    """Activations so small that d * xscale and the sums are subnormal, against
    the oracle; and smaller still, where 127 / amax overflows (the int8 codes
    then are what the conversion of an infinity gives), against the one-token
    kernels."""
    rows, cols = 70, 6144
    data = (quant_matrix(qtype, rows, cols, 970)[0] if qtype in (ref.Q4_K, ref.Q6_K, ref.Q8_0)
            else random_rows(qtype, rows, cols, 970))
    w = hip.Weight.from_host(data, qtype, rows, cols)
    xs = normal(971 + p, (p, cols), 5e-37)
    assert 0 < np.abs(xs).max() / 127 * 0.02 < np.finfo(np.float32).tiny
    got = w.matvec_batch(xs)
    assert np.any(got != 0)
    assert_bits(got, amd64(data, xs, rows, cols, qtype), f"type {qtype} p={p}")
    xs = normal(972 + p, (p, cols), 1e-38)
    one = np.stack([w.matvec_batch(x[None])[0] for x in xs])
    assert np.isfinite(one).all()
    assert_bits(w.matvec_batch(xs), one, f"type {qtype} p={p} vs one token")


def test_prefill_extremes_closed_form(hip):
    """TestAuditQ4KDotExtremes (q4k_q8_amd64_audit_test.go:18-52) batched: every
    code byte 0xff, d = dmin = 1, x = +-1 -> q8 = +-127, sc = m = 63, nibbles 15;
    per block 63 * 15 * 127 * 256 - 63 * 32 * 8 (x = +1)."""
    rows, cols, p = 48, 1024, 32
    blk = np.full(144, 0xFF, np.uint8)
    blk[0:2] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    blk[2:4] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    data = np.tile(blk, rows * (cols // 256))
    w = hip.Weight.from_host(data, ref.Q4_K, rows, cols)
    xs = np.where(np.arange(p)[:, None] % 2 == 0, 1.0, -1.0).astype(np.float32) * np.ones((p, cols),
                                                                                          np.float32)
    got = w.matvec_batch(xs)
    # the integer parts are exact; d * xscale = 1/127 rounds, hence rtol
    per_block = 63.0 * 15 * 256 - 63.0 * 32 * 8
    assert np.allclose(got[0::2], per_block * (cols // 256), rtol=1e-6)
    assert np.allclose(got[1::2], -per_block * (cols // 256), rtol=1e-6)
    assert_bits(got, amd64(data, xs, rows, cols), "extremes")


def device_weight(hip, qtype, rows, cols, seed):
    """Seeded N(0, 0.02) rows encoded on the device (the RTN encoders)."""
    import torch
    tmp = torch.empty((rows, cols), dtype=torch.float32, device="cuda")
    hip.fill_normal_dev(tmp, seed, 0.02)
    raw = torch.empty(rows * hip.row_bytes(qtype, cols), dtype=torch.uint8, device="cuda")
    hip.quantize_rows_dev(qtype, tmp, raw)
    del tmp
    return hip.Weight.from_device(raw, qtype, rows, cols), raw


@pytest.mark.parametrize("rows", [4096, 14336])
def test_prefill_configs2(hip, rows):
    """Q4_K rows x 4096 (seeded N(0, 0.02), device RTN encoder)
    against 512 activation rows N(0, 1): every token against the amd64-order
    oracle and against the GPU's own batch-1 path."""
    import torch
    cols, p = 4096, 512
    w, raw = device_weight(hip, hip.TYPE_Q4_K, rows, cols, 3000 + rows)
    x = torch.empty((p, cols), dtype=torch.float32, device="cuda")
    hip.fill_normal_dev(x, 77, 1.0)
    out = torch.empty((p, rows), dtype=torch.float32, device="cuda")
    print(f"prefill configs[2] {rows}x{cols} p={p}", flush=True)
    w.matvec_dev(x, out)
    one = torch.empty((p, rows), dtype=torch.float32, device="cuda")
    for t in range(p):
        w.matvec_dev(x[t:t + 1], one[t:t + 1])
    torch.cuda.synchronize()
    got, per_token = out.cpu().numpy(), one.cpu().numpy()
    assert np.isfinite(got).all() and float(np.std(got)) > 0.1
    assert_bits(got, per_token, "batched vs per-token row kernel")
    want = amd64(raw.cpu().numpy(), x.cpu().numpy(), rows, cols)
    assert_bits(got, want, "every token vs amd64 oracle")


# Q6_K batches of more than 16 tokens take the matrix-core tiles when the
# row has a multiple of 8 blocks (2048 columns and up); 1024 columns keep the
# row kernels (same bits either way)
@pytest.mark.parametrize("rows,cols,p", [(300, 2048, 17), (300, 2048, 33), (64, 2048, 100),
                                         (1000, 4096, 64), (70, 14336, 40), (130, 1024, 40)])
def test_prefill_q6k_bit_exact_small(hip, rows, cols, p):
    data, _ = quant_matrix(ref.Q6_K, rows, cols, 600 + p + rows)
    w = hip.Weight.from_host(data, ref.Q6_K, rows, cols)
    xs = normal(601 + p, (p, cols))
    print(f"prefill Q6_K {rows}x{cols} p={p}", flush=True)
    got = w.matvec_batch(xs)
    assert_bits(got, amd64(data, xs, rows, cols, ref.Q6_K), "vs amd64 oracle")


def test_prefill_q6k_extremes(hip):
    """Scales -128 and 127 with codes 63 (the largest |sc * code|, past f16's
    exact integers: the split at the code's fields keeps it exact), zero and
    large activations, against the oracle."""
    rows, cols, p = 64, 2048, 24
    rng = np.random.default_rng(91)
    data, _ = quant_matrix(ref.Q6_K, rows, cols, 92)
    blocks = data.reshape(rows * (cols // 256), 210)
    blocks[0::2, 0:192] = 0xFF                  # every code 63
    blocks[0::2, 192:208] = np.where(rng.random((len(blocks[0::2]), 16)) < 0.5, 0x80, 0x7F)
    blocks[1::4, 192:208] = 0x80                # scale -128 with random codes
    xs = normal(93, (p, cols))
    xs[0] = 0.0
    xs[1] *= 1e4
    xs[2, :] = np.where(np.arange(cols) % 2 == 0, 1.0, -1.0)
    w = hip.Weight.from_host(data, ref.Q6_K, rows, cols)
    got = w.matvec_batch(xs)
    assert_bits(got, amd64(data, xs, rows, cols, ref.Q6_K), "extremes vs amd64 oracle")


@pytest.mark.parametrize("rows,cols", [(14336, 4096), (4096, 14336)])
def test_prefill_q6k_configs2_shapes(hip, rows, cols):
    """Q6_K at the configs[1] / configs[2] shapes (a Q4_K_M file's ffn_down
    and attn_v are Q6_K), 512 tokens: every token against the amd64-order
    oracle."""
    import torch
    p = 512
    w, raw = device_weight(hip, hip.TYPE_Q6_K, rows, cols, 4000 + rows)
    x = torch.empty((p, cols), dtype=torch.float32, device="cuda")
    hip.fill_normal_dev(x, 78, 1.0)
    out = torch.empty((p, rows), dtype=torch.float32, device="cuda")
    print(f"prefill Q6_K {rows}x{cols} p={p}", flush=True)
    w.matvec_dev(x, out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.isfinite(got).all() and float(np.std(got)) > 0.1
    want = amd64(raw.cpu().numpy(), x.cpu().numpy(), rows, cols, ref.Q6_K)
    assert_bits(got, want, "every token vs amd64 oracle")


@pytest.mark.parametrize("rows,cols,p", [(300, 1024, 17), (64, 256, 100), (1000, 4096, 64),
                                         (70, 14336, 40), (130, 2048, 33)])
def test_prefill_q8_0_bit_exact_small(hip, rows, cols, p):
    """Q8_0 batches of more than 16 tokens: ragged row and token tiles against
    the amd64-order oracle."""
    data, _ = quant_matrix(ref.Q8_0, rows, cols, 700 + p + rows)
    w = hip.Weight.from_host(data, ref.Q8_0, rows, cols)
    xs = normal(701 + p, (p, cols))
    xs[0] = 0.0
    xs[1] *= 1e4
    print(f"prefill Q8_0 {rows}x{cols} p={p}", flush=True)
    got = w.matvec_batch(xs)
    assert_bits(got, amd64(data, xs, rows, cols, ref.Q8_0), "vs amd64 oracle")


def test_prefill_q8_0_extremes(hip):
    """Weights -128 and 127 against activations +-127: every 4-byte dot at
    its extremes (the reference's VPMADDUBSW pairs stay inside int16)."""
    rows, cols, p = 64, 1024, 20
    data, _ = quant_matrix(ref.Q8_0, rows, cols, 94)
    blocks = data.reshape(rows * (cols // 32), 34)
    blocks[0::2, 2:] = 0x80                     # -128
    blocks[1::2, 2:] = 0x7F                     # 127
    xs = np.where(np.arange(cols) % 3 == 0, 1.0, -1.0).astype(np.float32) * np.ones((p, 1), np.float32)
    xs[1::2] *= -1.0
    w = hip.Weight.from_host(data, ref.Q8_0, rows, cols)
    got = w.matvec_batch(xs)
    assert_bits(got, amd64(data, xs, rows, cols, ref.Q8_0), "extremes vs amd64 oracle")


@pytest.mark.parametrize("rows,cols", [(14336, 4096), (4096, 14336)])
def test_prefill_q8_0_configs2_shapes(hip, rows, cols):
    """Q8_0 at the configs[1] / configs[2] shapes, 512 tokens: every token
    against the amd64-order oracle."""
    import torch
    p = 512
    w, raw = device_weight(hip, hip.TYPE_Q8_0, rows, cols, 5000 + rows)
    x = torch.empty((p, cols), dtype=torch.float32, device="cuda")
    hip.fill_normal_dev(x, 79, 1.0)
    out = torch.empty((p, rows), dtype=torch.float32, device="cuda")
    print(f"prefill Q8_0 {rows}x{cols} p={p}", flush=True)
    w.matvec_dev(x, out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.isfinite(got).all() and float(np.std(got)) > 0.1
    want = amd64(raw.cpu().numpy(), x.cpu().numpy(), rows, cols, ref.Q8_0)
    assert_bits(got, want, "every token vs amd64 oracle")
