"""GPU parity: dequantisation (bit-exact) and the GEMV family (scaled error <= 5e-5, the engine's
own bar: native/tests/test_graph.cpp:45-52) through the C ABI, against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 5e-5  # |a - e| / max(1, |e|), native/src/main.cpp:165


def scaled_error(actual, expected):
    actual, expected = np.asarray(actual, dtype=np.float64), np.asarray(expected, dtype=np.float64)
    assert np.isfinite(actual).all()
    return float(np.max(np.abs(actual - expected) / np.maximum(1.0, np.abs(expected))))


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


# ---------------------------------------------------------------------------------- dequantise

def test_f16_all_patterns_bit_exact(gpu, orc):
    finite = np.array([b for b in range(65536) if (b >> 10) & 31 != 31], dtype=np.uint16)
    got = gpu.dequantize(1, gpu.upload(finite), finite.size).cpu().numpy()
    want = np.array([orc.binary16(int(b)) for b in finite], dtype=np.float32)
    assert np.array_equal(bits(got), bits(want)) and gpu.error() == 0
    inf = np.array([0x3C00, 0x7C00], dtype=np.uint16)
    gpu.dequantize(1, gpu.upload(inf), 2)
    assert gpu.error() == 1  # the reference refuses non-finite weights; the device flags them


@pytest.mark.parametrize("t", [0, 1, 7, 8, 12, 13, 14, 20, 30])
def test_dequantize_bit_exact_vs_oracle(gpu, orc, synth, t):
    epb, bpb = orc.encoding(t)
    nblocks = 4096 if epb > 1 else 40000
    if t in synth.BLOCKS:
        raw = synth.BLOCKS[t][0](1000 + t, nblocks).reshape(-1)
    elif t == 20:
        raw = synth.uniform_bytes(1020, nblocks * 18).reshape(nblocks, 18).copy()
        raw[:, 0:2] = synth.f16_bits(np.abs(synth.normal(1021, nblocks, 0.05))).view(np.uint8).reshape(nblocks, 2)
        raw = raw.reshape(-1)
    else:
        vals = synth.normal(1030 + t, nblocks, 3.0).astype(np.float32)
        raw = (vals.view(np.uint8) if t == 0 else synth.f16_bits(vals).view(np.uint8) if t == 1 else synth.bf16_bits(vals).view(np.uint8)).copy()
    want = orc.dequantize(t, raw, nblocks * epb)
    got = gpu.dequantize(t, gpu.upload(raw), nblocks * epb).cpu().numpy()
    assert np.array_equal(bits(got), bits(want)) and gpu.error() == 0


@pytest.mark.parametrize("t", [8, 12, 14])
def test_dequantize_edge_scales(gpu, orc, t):
    # native/tests/test_graph.cpp / test_metal.cpp scale set: zero, subnormal, +-0.25, 0x2800, plus f16 extremes.
    rng = np.random.default_rng(40 + t)
    epb, bpb = orc.encoding(t)
    scales = [0x0000, 0x8000, 0x0011, 0x0001, 0x03FF, 0x0400, 0x3400, 0xB400, 0x2800, 0x7BFF, 0xFBFF]
    raw = rng.integers(0, 256, size=(len(scales) * 8, bpb), dtype=np.uint8)
    for i in range(raw.shape[0]):
        s = scales[i % len(scales)]
        for off in ((0, 2) if t == 12 else (208,) if t == 14 else (0,)):
            raw[i, off], raw[i, off + 1] = s & 255, s >> 8
    n = raw.shape[0] * epb
    want = orc.dequantize(t, raw.reshape(-1), n)
    got = gpu.dequantize(t, gpu.upload(raw.reshape(-1)), n).cpu().numpy()
    assert np.array_equal(bits(got), bits(want)) and gpu.error() == 0


@pytest.mark.parametrize("t,cols,rows", [(12, 2048, 512), (13, 512, 64), (8, 512, 64), (7, 640, 32), (14, 512, 2048)])
def test_dequantize_planar_bit_exact(gpu, tsp, orc, synth, t, cols, rows):
    # native/tests/test_planar_pack_v3.cpp:269-275: planar dequant == GGUF dequant to the bit.
    raw = synth.matrix(t, 1100 + t, rows, cols)
    spec = tsp.make_expert_spec(t, cols, rows)
    planar = tsp.pack_expert(spec, raw)
    got = gpu.dequantize_planar(spec, gpu.upload(planar)).cpu().numpy()
    assert np.array_equal(bits(got), bits(orc.dequantize(t, raw, rows * cols))) and gpu.error() == 0


def test_dequantize_refusals(gpu, tsp):
    blocks = gpu.zeros(144, "uint8")
    with pytest.raises(tsp.FormatError):
        gpu.dequantize(12, blocks, 255)
    with pytest.raises(tsp.FormatError):
        gpu.dequantize(99, blocks, 256)


# ---------------------------------------------------------------------------------- GEMV

def reference_like_matrix(t, rows, cols, orc):
    """native/tests/test_graph.cpp:95-110: patterned bytes with fixed small scales."""
    epb, bpb = orc.encoding(t)
    data = np.array([(i * 37 + 19) & 255 for i in range(rows * (cols // epb) * bpb)], dtype=np.uint8).reshape(-1, bpb)
    for blk in data:
        if t == 0:
            blk[0:4] = np.frombuffer(np.float32(0.125).tobytes(), dtype=np.uint8)
        elif t == 30:
            blk[0:2] = (0x00, 0x3E)
        else:
            off = 208 if t == 14 else 0
            blk[off:off + 2] = (0x00, 0x24)
            if t in (7, 12, 13):
                blk[2:4] = (0x00, 0x20)
    return data.reshape(-1)


@pytest.mark.parametrize("t", [0, 1, 7, 8, 12, 13, 14, 20, 30])
def test_gemv_all_encodings_reference_fixture(gpu, orc, t):
    epb, _ = orc.encoding(t)
    cols, rows = epb * 3, 7
    w = reference_like_matrix(t, rows, cols, orc)
    x = np.array([((i % 31) - 15) / 16.0 for i in range(cols)], dtype=np.float32)
    want = orc.reference_gemv(t, w, cols, rows, x)
    dw, dx = gpu.upload(w), gpu.upload(x)
    for _ in range(3):
        got = gpu.gemv(t, dw, dx, cols, rows).cpu().numpy()
        assert scaled_error(got, want) <= TOL and gpu.error() == 0


@pytest.mark.parametrize("rows", [1, 3, 4, 5, 33])
@pytest.mark.parametrize("t,cols", [(12, 512), (12, 2048), (12, 4096), (12, 768), (14, 512), (8, 2048), (8, 96), (8, 4160)])
def test_gemv_shapes(gpu, orc, synth, t, cols, rows):
    w = synth.matrix(t, 1200 + t + rows, rows, cols)
    x = synth.activations_f32(1201, cols)
    want = orc.reference_gemv(t, w, cols, rows, x)
    got = gpu.gemv(t, gpu.upload(w), gpu.upload(x), cols, rows).cpu().numpy()
    assert scaled_error(got, want) <= TOL and gpu.error() == 0
    zero = gpu.gemv(t, gpu.upload(w), gpu.zeros(cols), cols, rows).cpu().numpy()
    assert not zero.any()  # zero input gives exactly zero output (native/tests/test_metal.cpp:41-66)


def test_config0_dense_q4k_gemv(gpu, tsp, orc, synth):
    """BASELINE config 0 at full size: W 4096 x 2048 Q4_K, x f32 N(0,1); raw GGUF rows and planar v3."""
    rows, cols = 4096, 2048
    w = synth.matrix(12, synth.tensor_seed(0, 1), rows, cols)
    x = synth.activations_f32(synth.tensor_seed(0, 2), cols)
    want = orc.reference_gemv_mt(12, w, cols, rows, x, 8)
    dx = gpu.upload(x)
    got = gpu.gemv(12, gpu.upload(w), dx, cols, rows).cpu().numpy()
    err_raw = scaled_error(got, want)
    spec = tsp.make_expert_spec(12, cols, rows)
    planar = tsp.pack_expert(spec, w)
    got_p = gpu.gemv(12, gpu.upload(planar), dx, cols, rows, layout=tsp.LAYOUT_PLANAR_V3).cpu().numpy()
    assert gpu.error() == 0
    # the two arms share their arithmetic: identical bits (the engine's block path is held to this too,
    # native/tests/test_block_gemv.cpp:94)
    assert np.array_equal(bits(got), bits(got_p))
    # The configuration's bar is max scaled error 2e-3 with f32 accumulation. Measured: 6.2e-5, on an element of magnitude ~1
    # in a vector whose entries reach several hundred (weights up to ~19, 2048 products): 3e-7 of the vector's scale, which
    # is what f32 accumulation leaves. The engine's 5e-5 (native/src/main.cpp:165) is quoted on outputs of magnitude ~1 and
    # holds at those (test_gemv_shapes, test_gemv_all_encodings_reference_fixture); here the bound asserted is 2e-4.
    print(f"config0 max scaled error {err_raw:.3e}")
    assert err_raw <= 2e-4, err_raw


def test_gemv_rows_strided(gpu, orc, synth):
    # include/tokspur/graph.hpp:733: gemv once per row of a strided row set; padding stays untouched.
    cols, rows, count = 2048, 64, 5
    w = synth.matrix(12, 1300, rows, cols)
    x = synth.activations_f32(1301, (count, cols + 8))
    y = gpu.full((count, rows + 4), -7.0)
    gpu.gemv_rows(12, gpu.upload(w), gpu.upload(x), y, count, cols, rows, (cols + 8) * 4, (rows + 4) * 4)
    y = y.cpu().numpy()
    for i in range(count):
        assert scaled_error(y[i, :rows], orc.reference_gemv(12, w, cols, rows, x[i, :cols])) <= TOL
    assert (y[:, rows:] == -7.0).all() and gpu.error() == 0


@pytest.mark.parametrize("t", [0, 1, 7, 8, 12, 13, 14, 20, 30])
def test_routed_gemv(gpu, orc, synth, t):
    # native/tests/test_moe.cpp:96-129: per selected expert, both broadcast and per-route inputs.
    epb, bpb = orc.encoding(t)
    cols, rows, experts, selected = epb * 2 if epb > 1 else 64, 9, 6, 4
    w = np.concatenate([reference_like_matrix(t, rows, cols, orc)[::1] for _ in range(experts)])
    w = w.copy()
    rng = np.random.default_rng(t)
    per = w.size // experts
    for e in range(experts):  # make experts differ in their quant bytes, keep the scale fields
        blk = w[e * per:(e + 1) * per].reshape(-1, bpb)
        lo = 4 if t in (7, 12, 13) else 2 if t in (8, 20, 1, 30) else 0
        hi = 208 if t == 14 else bpb
        if epb > 1:
            blk[:, lo:hi] = rng.integers(0, 256, size=(blk.shape[0], hi - lo), dtype=np.uint8)
    ids = np.array([5, 0, 3, 5], dtype=np.uint32)
    for broadcast in (True, False):
        x = synth.activations_f32(1400 + t, (1 if broadcast else selected, cols))
        got = gpu.routed_gemv(t, gpu.upload(w), gpu.upload(ids), gpu.upload(x), cols, rows, experts, selected, broadcast).cpu().numpy()
        for s, e in enumerate(ids):
            want = orc.reference_gemv(t, w[e * per:(e + 1) * per], cols, rows, x[0 if broadcast else s])
            assert scaled_error(got[s], want) <= TOL
        assert gpu.error() == 0


def test_sticky_error_word(gpu, tsp, orc, synth):
    # native/tests/test_moe.cpp:165-190: non-finite input or bad id poisons the batch; the next batch is clean.
    cols, rows = 2048, 16
    w = synth.matrix(12, 1500, rows, cols)
    x = synth.activations_f32(1501, cols)
    dw = gpu.upload(w)
    bad = x.copy()
    bad[7] = np.inf
    gpu.gemv(12, dw, gpu.upload(bad), cols, rows)
    assert gpu.error() & tsp.ERRBIT_NONFINITE
    got = gpu.gemv(12, dw, gpu.upload(x), cols, rows).cpu().numpy()
    assert gpu.error() == 0 and scaled_error(got, orc.reference_gemv(12, w, cols, rows, x)) <= TOL
    ids = gpu.upload(np.array([0, 9], dtype=np.uint32))
    wq = gpu.upload(synth.matrix(8, 1502, 4 * 2, 64))
    out = gpu.routed_gemv(8, wq, ids, gpu.upload(synth.activations_f32(1503, 64)), 64, 4, 2, 2, True).cpu().numpy()
    assert gpu.error() & tsp.ERRBIT_INDEX and not out[1].any()


def test_gemv_refusals(gpu, tsp, synth):
    w = gpu.upload(synth.matrix(12, 1600, 4, 256))
    x, y = gpu.zeros(256), gpu.zeros(4)
    for args in ((12, w, x, 256, 5), (12, w, x, 255, 4), (99, w, x, 256, 4), (12, w, x, 0, 4)):
        with pytest.raises(tsp.FormatError):
            gpu.gemv(*args)
    with pytest.raises(tsp.FormatError):  # output aliasing an input
        gpu.gemv(0, x, x, 16, 16, y=x)


# ---------------------------------------------------------------------------------- Q8 many rows

@pytest.mark.parametrize("tokens,cols,rows", [(1, 64, 5), (19, 512, 160), (40, 2048, 96), (9, 1024, 64), (13, 2048, 1000), (16, 2048, 2084),
                                              (27, 1024, 132), (8, 1536, 77), (3, 512, 16)])
def test_dense_mm_q8(gpu, tsp, orc, synth, tokens, cols, rows):
    # graph.hpp:860 `dense_mm_q8`: a dense Q8_0 matrix times f32 rows, GGUF rows and q8_lanes_v1 rows; rows back to back
    # (width groups 8, 4, 2, 1; nine or more GGUF rows of 1024 / 2048 columns go up to sixteen at a time, each half of the
    # columns summed by its own workgroups) and rows with padding (canaries stay)
    w = synth.matrix(8, 1800 + cols, rows, cols)
    lanes = tsp.q8_lanes_pack_rows(cols, w)
    x = synth.activations_f32(1801 + tokens, (tokens, cols + 4))
    want = np.stack([orc.reference_gemv(8, w, cols, rows, x[t, :cols]) for t in range(tokens)])
    for matrix, layout in ((w, tsp.LAYOUT_GGUF), (lanes, tsp.LAYOUT_Q8_LANES_V1)):
        packed = tsp.dense_mm_q8(gpu, layout, gpu.upload(matrix), gpu.upload(np.ascontiguousarray(x[:, :cols])), tokens, cols, rows).cpu().numpy()
        assert scaled_error(packed, want) <= TOL and gpu.error() == 0
        out = gpu.full((tokens, rows + 3), -5.0)
        tsp.dense_mm_q8(gpu, layout, gpu.upload(matrix), gpu.upload(x), tokens, cols, rows, out=out, x_stride=(cols + 4) * 4, out_stride=(rows + 3) * 4)
        got = out.cpu().numpy()
        assert scaled_error(got[:, :rows], want) <= TOL and (got[:, rows:] == -5.0).all() and gpu.error() == 0
    with pytest.raises(tsp.FormatError):
        tsp.dense_mm_q8(gpu, tsp.LAYOUT_PLANAR_V3, gpu.upload(w), gpu.upload(x), tokens, cols, rows, x_stride=(cols + 4) * 4)


@pytest.mark.parametrize("tokens,cols,rows", [(1, 64, 5), (70, 128, 33), (200, 2048, 512), (129, 512, 2048), (64, 4096, 64), (45, 1088, 30)])
def test_dense_mm_q8_staged(gpu, tsp, orc, synth, tokens, cols, rows):
    # the many-row form of graph.hpp:860 `dense_mm_q8`: matrix and rows as halves, one matrix-core GEMM. Both layouts, rows with
    # padding on both sides (canaries stay), tiles that overhang the matrix on either edge, and agreement with the streaming
    # entry point.
    w = synth.matrix(8, 1900 + cols, rows, cols)
    lanes = tsp.q8_lanes_pack_rows(cols, w)
    x = synth.activations_f32(1901 + tokens, (tokens, cols + 4))
    sample = np.unique(np.linspace(0, tokens - 1, min(tokens, 24)).astype(int))
    want = np.stack([orc.reference_gemv(8, w, cols, rows, x[t, :cols]) for t in sample])
    scale = np.maximum(1.0, np.sqrt((want ** 2).mean(axis=1, keepdims=True)))
    streamed = tsp.dense_mm_q8(gpu, tsp.LAYOUT_GGUF, gpu.upload(w), gpu.upload(np.ascontiguousarray(x[:, :cols])), tokens, cols, rows).cpu().numpy()
    for matrix, layout in ((w, tsp.LAYOUT_GGUF), (lanes, tsp.LAYOUT_Q8_LANES_V1)):
        out = gpu.full((tokens, rows + 3), -5.0)
        tsp.dense_mm_q8_staged(gpu, layout, gpu.upload(matrix), gpu.upload(x), tokens, cols, rows, out=out, x_stride=(cols + 4) * 4,
                               out_stride=(rows + 3) * 4)
        got = out.cpu().numpy()
        assert gpu.error() == 0 and (got[:, rows:] == -5.0).all()
        assert float(np.max(np.abs(got[sample, :rows] - want) / np.maximum(scale, np.abs(want)))) <= 2e-3  # the GEMM tolerance
        row_scale = np.maximum(1.0, np.sqrt((streamed ** 2).mean(axis=1, keepdims=True)))
        assert float(np.max(np.abs(got[:, :rows] - streamed) / np.maximum(row_scale, np.abs(streamed)))) <= 2e-3
        nmse = float(((got[:, :rows] - streamed) ** 2).sum() / max((streamed ** 2).sum(), 1e-30))
        assert nmse <= 1e-6, nmse
    with pytest.raises(tsp.FormatError):  # columns not a multiple of 64
        tsp.dense_mm_q8_staged(gpu, tsp.LAYOUT_GGUF, gpu.upload(synth.matrix(8, 3, 4, 96)), gpu.zeros((2, 96)), 2, 96, 4)
    with pytest.raises(tsp.FormatError):  # workspace too small
        tsp.dense_mm_q8_staged(gpu, tsp.LAYOUT_GGUF, gpu.upload(w), gpu.upload(x), tokens, cols, rows, x_stride=(cols + 4) * 4,
                               workspace=gpu.empty(256, "uint8"))
    x_bad = np.ascontiguousarray(x[:, :cols]).copy()
    x_bad[tokens // 2, cols // 2] = np.inf
    tsp.dense_mm_q8_staged(gpu, tsp.LAYOUT_GGUF, gpu.upload(w), gpu.upload(x_bad), tokens, cols, rows)
    assert gpu.error() & tsp.ERRBIT_NONFINITE
    gpu.clear_error()


@pytest.mark.parametrize("tokens,cols,rows", [(33, 2048, 31), (31, 2112, 65), (2, 64, 1), (65, 576, 33), (96, 192, 6400), (97, 64, 6401)])
def test_dense_mm_q8_staged_tiles(gpu, tsp, synth, tokens, cols, rows):
    # one tile and many, fewer steps than waves, a half step at the end, ragged tiles on both sides (which kernel has which call: test_dense_mm_q8_staged_kernels).
    # A weight and an activation are rounded to halves: 2^-11 each, so 2^-10 of the sum of |w| |x|.
    w = synth.matrix(8, 2400 + cols, rows, cols)
    x = synth.activations_f32(2401 + tokens, (tokens, cols))
    got = tsp.dense_mm_q8_staged(gpu, tsp.LAYOUT_GGUF, gpu.upload(w), gpu.upload(x), tokens, cols, rows).cpu().numpy()
    blocks = w.reshape(rows, -1, 34)
    weight = blocks[:, :, 2:].view(np.int8).astype(np.float64) * np.ascontiguousarray(blocks[:, :, :2]).view(np.float16).astype(np.float64)
    weight = weight.reshape(rows, cols)
    bound = (2.0 ** -10 + cols * 2.0 ** -24) * (np.abs(x.astype(np.float64)) @ np.abs(weight).T)
    assert (np.abs(got - x.astype(np.float64) @ weight.T) <= bound).all() and gpu.error() == 0


@pytest.mark.parametrize("tokens,cols,rows,pad", [(33, 64, 33, 0), (63, 2624, 31, 1), (100, 704, 2500, 0), (203, 704, 2500, 3), (2043, 2112, 701, 0), (1990, 704, 2040, 1),
                                                  (449, 640, 2500, 0)])
def test_dense_mm_q8_staged_tile_shapes(gpu, tsp, synth, tokens, cols, rows, pad):
    # every tile that raw rows are decoded in (32 x 32, 32 x 32, 32 x 64, 64 x 64, 64 x 96, 128 x 128) and the two launches: ragged edges, a last step of 64 columns, a single
    # step, rows four bytes off a multiple of sixteen. The bound is that of test_dense_mm_q8_staged_tiles.
    w = synth.matrix(8, 2500 + cols, rows, cols)
    x = synth.activations_f32(2501 + tokens, (tokens, cols + pad))
    out = gpu.full((tokens, rows + 3), -5.0)
    tsp.dense_mm_q8_staged(gpu, tsp.LAYOUT_GGUF, gpu.upload(w), gpu.upload(x), tokens, cols, rows, out=out, x_stride=(cols + pad) * 4, out_stride=(rows + 3) * 4)
    got, x = out.cpu().numpy(), x[:, :cols].astype(np.float64)
    blocks = w.reshape(rows, -1, 34)
    weight = blocks[:, :, 2:].view(np.int8).astype(np.float64) * np.ascontiguousarray(blocks[:, :, :2]).view(np.float16).astype(np.float64)
    weight = weight.reshape(rows, cols)
    bound = (2.0 ** -10 + cols * 2.0 ** -24) * (np.abs(x) @ np.abs(weight).T)
    assert (np.abs(got[:, :rows] - x @ weight.T) <= bound).all() and (got[:, rows:] == -5.0).all() and gpu.error() == 0


@pytest.mark.parametrize("tokens,cols,rows,kernels", [(63, 2624, 31, ["q8_gemm_fused 32x32"]), (100, 704, 2500, ["q8_gemm_fused 32x64"]), (203, 704, 2500, ["q8_gemm_fused 64x64"]),
                                                      (2043, 1088, 701, ["q8_gemm_fused 64x96"]), (1990, 704, 2040, ["q8_gemm_fused 128x128"]), (70, 128, 33, ["q8_gemm_split"]), (9, 2624, 33, ["q8_gemm_split"]),
                                                      (1990, 704, 1021, ["q8_operands_to_f16", "f16_gemm_nt"])])
def test_dense_mm_q8_staged_kernels(gpu, tsp, synth, tokens, cols, rows, kernels):
    # Which kernels a call takes, so that each is reached whatever the rule's figures; and in each an infinity and a finite value that
    # no half holds, one of them in the last token row's last 64 columns, are reported and leave all other token rows right (the bound of test_dense_mm_q8_staged_tiles).
    w = synth.matrix(8, 2600 + cols, rows, cols)
    x = synth.activations_f32(2601 + tokens, (tokens, cols))
    blocks = w.reshape(rows, -1, 34)
    weight = blocks[:, :, 2:].view(np.int8).astype(np.float64) * np.ascontiguousarray(blocks[:, :, :2]).view(np.float16).astype(np.float64)
    weight = weight.reshape(rows, cols)
    declared, bound = x.astype(np.float64) @ weight.T, (2.0 ** -10 + cols * 2.0 ** -24) * (np.abs(x.astype(np.float64)) @ np.abs(weight).T)
    matrix = gpu.upload(w)
    tsp.profile_begin()
    got = tsp.dense_mm_q8_staged(gpu, tsp.LAYOUT_GGUF, matrix, gpu.upload(x), tokens, cols, rows).cpu().numpy()
    assert sorted(tsp.profile_end()) == sorted(kernels)
    assert (np.abs(got - declared) <= bound).all() and gpu.error() == 0
    for at, value in ((tokens - 1, np.inf), (tokens - 1, 1e5), (tokens // 2, -np.inf), (tokens // 2, -1e5)):
        wrong = x.copy()
        wrong[at, cols - 3 if at == tokens - 1 else 1] = value
        got = tsp.dense_mm_q8_staged(gpu, tsp.LAYOUT_GGUF, matrix, gpu.upload(wrong), tokens, cols, rows).cpu().numpy()
        assert gpu.error() & tsp.ERRBIT_NONFINITE
        gpu.clear_error()
        others = np.arange(tokens) != at
        assert (np.abs(got - declared) <= bound)[others].all()


@pytest.mark.parametrize("tokens,cols,rows,pad,kernels", [
    (400, 64, 640, 0, "split"), (9, 320, 33, 0, "split"), (601, 64, 1601, 0, "split"), (561, 64, 1601, 1, "64x64"), (1001, 64, 1601, 0, "two"), (33, 64, 33, 1, "two"), (700, 192, 1000, 0, "64x64"), (33, 384, 33, 0, "32x32"), (1600, 384, 700, 0, "two"),       # few columns; rows that the first cannot read
    (1, 2048, 33, 0, "split"), (16, 4096, 65, 4, "split"), (16, 2048, 65, 3, "32x32"), (17, 2048, 65, 0, "32x32"), (16, 1024, 65, 0, "32x32"),  # few tokens
    (700, 2112, 1024, 0, "two"), (250, 2112, 3100, 0, "64x64"), (1025, 1024, 512, 0, "64x64"), (1025, 1088, 512, 0, "two"), (820, 1088, 512, 0, "32x64"), (1200, 2112, 512, 0, "two")])
def test_dense_mm_q8_staged_choice(gpu, tsp, synth, tokens, cols, rows, pad, kernels):
    # Calls that the rule by rounds over the chip alone had made up to 1.5 times as long as they were (few columns, few tokens) or 1.1 times (many columns from memory), and
    # either side of its limits. The bound is that of test_dense_mm_q8_staged_tiles.
    w = synth.matrix(8, 2700 + cols, rows, cols)
    x = synth.activations_f32(2701 + tokens, (tokens, cols + pad))
    matrix, rows_in = gpu.upload(w), gpu.upload(x)
    tsp.profile_begin()
    got = tsp.dense_mm_q8_staged(gpu, tsp.LAYOUT_GGUF, matrix, rows_in, tokens, cols, rows, x_stride=(cols + pad) * 4).cpu().numpy()
    assert sorted(tsp.profile_end()) == {"split": ["q8_gemm_split"], "two": ["f16_gemm_nt", "q8_operands_to_f16"]}.get(kernels, ["q8_gemm_fused " + kernels])
    x = x[:, :cols].astype(np.float64)
    blocks = w.reshape(rows, -1, 34)
    weight = blocks[:, :, 2:].view(np.int8).astype(np.float64) * np.ascontiguousarray(blocks[:, :, :2]).view(np.float16).astype(np.float64)
    weight = weight.reshape(rows, cols)
    bound = (2.0 ** -10 + cols * 2.0 ** -24) * (np.abs(x) @ np.abs(weight).T)
    assert (np.abs(got - x @ weight.T) <= bound).all() and gpu.error() == 0


@pytest.mark.parametrize("tokens,cols,rows,pad", [(2, 64, 1, 0), (7, 640, 33, 0), (8, 2560, 640, 0), (9, 320, 18, 0), (16, 1088, 47, 12), (5, 2048, 160, 4),
                                                  (23, 2560, 48, 0), (3, 96, 20, 0), (6, 512, 24640, 0), (15, 512, 14020, 0), (11, 1280, 14001, 0),
                                                  (7, 2560, 24577, 0), (14, 2560, 14004, 0), (27, 1024, 14004, 0), (41, 192, 30, 4),
                                                  (18, 768, 6144, 0), (18, 768, 6145, 0), (64, 2048, 7000, 0), (64, 2048, 8200, 0), (8, 1536, 12288, 0), (37, 512, 10300, 0),
                                                  (18, 768, 12288, 0), (18, 768, 12289, 0), (64, 2048, 7200, 0), (64, 2048, 9217, 0), (40, 1280, 11400, 0), (33, 2304, 17000, 0)])
def test_dense_mm_q8_few_rows(gpu, tsp, orc, synth, tokens, cols, rows, pad):
    # every kernel that a few raw Q8_0 token rows can go to: 16-row tiles (any multiple of 64 columns, rows any distance apart), or, up to sixteen at a time,
    # the persistent ones, from 6000 to 31 000 rows on; either side of where a pass of those and what is left over take the place of the tiles
    w = synth.matrix(8, 2200 + cols, rows, cols)
    x = synth.activations_f32(2201 + tokens, (tokens, cols + pad))
    x[0] *= 1e-20
    x[-1] *= 1e4
    check = np.unique(np.r_[0:min(rows, 40), max(0, rows - 40):rows])
    part = np.ascontiguousarray(w.reshape(rows, -1)[check]).reshape(-1)
    want = np.stack([orc.reference_gemv(8, part, cols, len(check), np.ascontiguousarray(x[t, :cols])) for t in range(tokens)])
    out = gpu.full((tokens, rows + pad), -5.0)
    tsp.dense_mm_q8(gpu, tsp.LAYOUT_GGUF, gpu.upload(w), gpu.upload(x), tokens, cols, rows, out=out, x_stride=(cols + pad) * 4, out_stride=(rows + pad) * 4)
    got = out.cpu().numpy()
    # against the sum of |w| |x|: 2^-22 for the two halves of an activation, and a few 2^-24 for each rounding on the way through
    # 32-column sums and their addition; where halves are subnormal under the row's power of two, 2^-38 of its largest
    blocks = part.reshape(len(check), -1, 34)
    weight = np.abs(blocks[:, :, 2:].view(np.int8).astype(np.float64)) * np.ascontiguousarray(blocks[:, :, :2]).view(np.float16).astype(np.float64)
    weight = weight.reshape(len(check), cols)
    bound = 2.0 ** -19 * (np.abs(x[:, :cols].astype(np.float64)) @ weight.T) + 2.0 ** -38 * np.abs(x).max(axis=1, keepdims=True) * weight.sum(1)
    assert (np.abs(got[:, check] - want) <= bound).all() and (got[:, rows:] == -5.0).all() and gpu.error() == 0


@pytest.mark.parametrize("width", [1, 2, 4, 8])
@pytest.mark.parametrize("cols,rows", [(2048, 37), (64, 5), (96, 7), (4096, 9)])
def test_q8_matvec_many(gpu, tsp, orc, synth, width, cols, rows):
    # native/tests/test_q8_many.cpp: token-major in and out, every width, both layouts.
    w = synth.matrix(8, 1700 + cols, rows, cols)
    x = synth.activations_f32(1701 + width, (width, cols))
    want = orc.reference_q8_many(w, x, cols, rows, width)
    got = gpu.q8_matvec_many(gpu.upload(w), gpu.upload(x), cols, rows, width).cpu().numpy()
    assert scaled_error(got, want) <= TOL and gpu.error() == 0
    lanes = tsp.q8_lanes_pack_rows(cols, w)
    got_l = gpu.q8_matvec_many(gpu.upload(lanes), gpu.upload(x), cols, rows, width, layout=tsp.LAYOUT_Q8_LANES_V1).cpu().numpy()
    assert scaled_error(got_l, want) <= TOL and gpu.error() == 0
    with pytest.raises(tsp.FormatError):
        gpu.q8_matvec_many(gpu.upload(w), gpu.upload(x), cols, rows, 3)


@pytest.mark.parametrize("cols,rows,count", [(4, 1, 3), (252, 5, 2), (2048, 512, 1), (2052, 3, 1), (2560, 1, 9), (4100, 2, 2), (2046, 3, 2)])
def test_gemv_f32_rows(gpu, synth, cols, rows, count):
    """Float rows in 16-byte pieces: fewer pieces than lanes, a second batch of 2048 columns, many token rows against one
    matrix row; 2046 columns stay with the per-element kernel. Error bound: f32 sums in any order, n/64 + 8 roundings."""
    w, x = synth.activations_f32(1900 + cols, (rows, cols)), synth.activations_f32(1901 + cols, (count, cols))
    y = gpu.empty((count, rows))
    gpu.gemv_rows(0, gpu.upload(w.view(np.uint8)), gpu.upload(x), y, count, cols, rows, cols * 4, rows * 4)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    scale = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    assert (np.abs(y.cpu().numpy() - want) <= (cols / 64 + 8) * 2.0 ** -24 * scale).all() and gpu.error() == 0


def zero_columns(t, raw, rows, cols):
    """Makes the sixth of every 32 weights of a GGUF matrix zero (Q4_K: the minima as well)."""
    blocks = raw.reshape(rows * cols // (32 if t == 8 else 256), -1)
    if t == 8:
        blocks[:, 7] = 0
    elif t == 12:
        blocks[:, 2:4] = 0
        blocks[:, 16 + 5:16 + 128:32] = 0  # both nibbles: the sixth of a pair's first and second 32
    else:
        blocks[:, [5, 37, 69, 101]] = 0  # low nibbles of elements 5, 37, 69, 101 of either section; the code 32 is zero
        blocks[:, [133, 165]] = 0xaa


@pytest.mark.parametrize("t,cols,rows", [(12, 256, 3), (12, 768, 70), (12, 2560, 513), (12, 6144, 9), (14, 256, 1), (14, 2560, 700), (14, 1280, 5000), (14, 12288, 2),
                                         (8, 32, 2), (8, 544, 33), (8, 2560, 600), (8, 5120, 17), (8, 1024, 9000)])
def test_gemv_units(gpu, orc, synth, t, cols, rows):
    """Rows of any length, 8 to 64 lanes per row, last rounds with idle lanes, more steps than waves. Error bound: a weight is rounded
    once, a product passes at most 16 roundings in its chain, 26 over a row's rounds and 6 across lanes: 2^-18 of sum |w x|.
    A second row of activations puts 3e4 to 1e30 in front of weights that are zero, one in each 32: nothing may be lost beside them."""
    w = synth.matrix(t, 2100 + cols, rows, cols)
    zero_columns(t, w, rows, cols)
    x = synth.activations_f32(2101 + rows, cols)
    x[cols // 2:] *= np.float32(1e-3)
    dense = orc.dequantize(t, w, rows * cols).reshape(rows, cols).astype(np.float64)
    assert not dense[:, 5::32].any()
    beside = x.copy()
    beside[5::32] = np.resize(np.array([3e4, -1e12, 1e30], dtype=np.float32), cols // 32)
    for values in (x, beside):
        bound = (np.abs(dense) @ np.abs(values.astype(np.float64))) * 2.0 ** -18
        got = gpu.gemv(t, gpu.upload(w), gpu.upload(values), cols, rows).cpu().numpy().astype(np.float64)
        assert (np.abs(got - dense @ values.astype(np.float64)) <= bound).all() and gpu.error() == 0
    x[1] = np.nan
    gpu.gemv(t, gpu.upload(w), gpu.upload(x), cols, rows)
    assert gpu.error() == 1


@pytest.mark.parametrize("t,cols", [(12, 512), (12, 2048), (12, 2560), (14, 512), (14, 2560), (8, 2048), (8, 2560)])
@pytest.mark.parametrize("exponent", [-70, -103, -110, -124])
def test_gemv_tiny_activations(gpu, orc, synth, t, cols, exponent):
    """Activations far below one, down to the smallest floats, multiply like any others. Error bound: as for test_gemv_units, and
    an f32 operation on subnormals is off by up to 2^-150 whatever its result: a few for each of the row's products."""
    rows = 65
    w = synth.matrix(t, 2500 + cols, rows, cols)
    x = synth.activations_f32(2501, cols) * np.float32(2.0 ** exponent)
    x[32:64] *= np.float32(2.0 ** -20)  # a sub-block of subnormals among the last exponent's
    x[64:96] = 0
    dense = orc.dequantize(t, w, rows * cols).reshape(rows, cols).astype(np.float64)
    bound = (np.abs(dense) * np.abs(x.astype(np.float64).reshape(-1, 32)).max(axis=1).repeat(32)).sum(axis=1) * (2.0 ** -23 + 2.0 ** -22) + cols * 2.0 ** -147
    got = gpu.gemv(t, gpu.upload(w), gpu.upload(x), cols, rows).cpu().numpy().astype(np.float64)
    assert (np.abs(got - dense @ x.astype(np.float64)) <= bound).all() and gpu.error() == 0


@pytest.mark.parametrize("lanes,tokens,cols,rows,pad", [(False, 2, 64, 1, 0), (False, 7, 640, 33, 0), (False, 8, 2560, 640, 0), (False, 9, 320, 18, 0), (False, 16, 1088, 47, 12),
                                                        (False, 5, 2048, 160, 4), (False, 21, 512, 30, 4), (False, 1, 2560, 40004, 0), (False, 5, 2560, 60001, 0),
                                                        (False, 8, 2560, 60000, 0), (False, 16, 2560, 25000, 0), (False, 13, 2304, 60000, 0), (True, 1, 2560, 16, 0), (True, 5, 2560, 1003, 0),
                                                        (True, 8, 2560, 4100, 0), (True, 16, 2560, 512, 0)])
def test_dense_mm_q8_f32_rows(gpu, tsp, orc, synth, lanes, tokens, cols, rows, pad):
    """Few token rows of up to 16 rows' tiles, and any of more than 2048 columns, are multiplied as the floats they are: 3e4 to 1e30 in front
    of weights that are zero, one in each 32, take nothing from the values beside them, nor does one row from another. Error
    bound: a block's sum in at most 12 roundings, 80 blocks or waves' sums one each: less than 2^-17 of sum |w x|."""
    w = synth.matrix(8, 2600 + cols, rows, cols)
    zero_columns(8, w, rows, cols)
    x = synth.activations_f32(2601 + tokens, (tokens, cols + pad))
    x[:, 5:cols:32] = np.resize(np.array([3e4, -1e12, 1e30], dtype=np.float32), (tokens, cols // 32))
    x[0] *= np.float32(1e-37) if tokens > 1 else np.float32(1)
    matrix = tsp.q8_lanes_pack_rows(cols, w) if lanes else w
    check = np.unique(np.r_[0:min(rows, 300), np.linspace(0, rows - 1, 500).astype(int), max(0, rows - 40):rows])
    dense = orc.dequantize(8, np.ascontiguousarray(w.reshape(rows, -1)[check]).reshape(-1), len(check) * cols).reshape(len(check), cols).astype(np.float64)
    out = gpu.full((tokens, rows + pad), -5.0)
    tsp.dense_mm_q8(gpu, tsp.LAYOUT_Q8_LANES_V1 if lanes else tsp.LAYOUT_GGUF, gpu.upload(matrix), gpu.upload(x), tokens, cols, rows, out=out,
                    x_stride=(cols + pad) * 4, out_stride=(rows + pad) * 4)
    got, x = out.cpu().numpy(), x[:, :cols].astype(np.float64)
    bound = 2.0 ** -17 * (np.abs(x) @ np.abs(dense).T) + cols * 2.0 ** -149
    assert gpu.error() == 0 and (got[:, rows:] == -5.0).all()
    assert (np.abs(got[:, check] - x @ dense.T) <= bound).all(), float(np.max(np.abs(got[:, check] - x @ dense.T) / bound))
    x = np.ascontiguousarray(x, dtype=np.float32)
    x[tokens // 2, cols - 1] = np.nan
    tsp.dense_mm_q8(gpu, tsp.LAYOUT_Q8_LANES_V1 if lanes else tsp.LAYOUT_GGUF, gpu.upload(matrix), gpu.upload(x), tokens, cols, rows)
    assert gpu.error() == tsp.ERRBIT_NONFINITE


@pytest.mark.parametrize("tokens,rows", [(6, 20), (7, 1002), (10, 1008), (11, 16), (15, 4112)])
def test_dense_mm_q8_lanes_half_rows(gpu, tsp, orc, synth, tokens, rows):
    """Six to ten rows of 2560 columns, two workgroups to a matrix row with its middle run shared, a last tile of four rows, an output whose length is no
    multiple of four; more than ten, ten waves to a matrix row. The bound of the test above: one more addition."""
    test_dense_mm_q8_f32_rows(gpu, tsp, orc, synth, True, tokens, 2560, rows, 0)


# one wave to ten, just past the sizes that a workgroup per sixteen rows takes and up to the last of floats; from five waves on some workgroups have a second
# tile or more, and most last tiles are of one row or a few (rounds of tiles: test_dense_mm_q8_resident_rounds)
@pytest.mark.parametrize("lanes,tokens,cols,rows", [(False, 2, 256, 12289), (False, 9, 512, 6001), (False, 16, 768, 6017), (False, 8, 1024, 16385), (False, 11, 1280, 8193),
                                                    (False, 16, 1536, 6001), (False, 10, 1792, 6016), (False, 5, 2048, 12321), (False, 7, 2304, 20481), (False, 16, 2560, 13003),
                                                    (True, 11, 2560, 17), (True, 16, 2560, 8193), (False, 9, 1792, 14016), (False, 16, 768, 14001), (False, 11, 1280, 20003),
                                                    (False, 13, 256, 24575)])
def test_dense_mm_q8_resident_rows(gpu, tsp, orc, synth, lanes, tokens, cols, rows):
    """Token rows in registers, a wave per 256 columns, as the floats they are: the bound of the tests above, ten waves' sums one addition each."""
    test_dense_mm_q8_f32_rows(gpu, tsp, orc, synth, lanes, tokens, cols, rows, 0)


@pytest.mark.parametrize("tokens,cols,rows", [(2, 256, 24577), (16, 768, 24577), (7, 1280, 24610), (9, 1792, 24600), (16, 2048, 16385)])
def test_dense_mm_q8_resident_halves(gpu, tsp, orc, synth, tokens, cols, rows):
    """The same of large matrices, in two halves under a power of two per row: the bound and the canaries of the test below."""
    test_dense_mm_q8_odd_rows(gpu, tsp, orc, synth, False, tokens, cols, rows)


@pytest.mark.parametrize("lanes,tokens,cols,rows", [(False, 2, 256, 24577), (False, 16, 768, 24577), (False, 7, 1280, 24610), (False, 9, 1792, 24600), (False, 16, 2048, 16385),
                                                    (False, 8, 2048, 24600), (True, 5, 512, 1001), (True, 16, 1024, 1000), (True, 8, 1536, 403), (True, 11, 2048, 1001)])
def test_dense_mm_q8_halves_far_apart(gpu, tsp, orc, synth, lanes, tokens, cols, rows):
    """Token rows in two halves each have a power of two of their own: rows of 1e-20 and 1e4 beside one another keep their bits. Error bound: as above for
    sums, and 22 bits of the row's largest value, or less where a half is subnormal: 2^-22 of each |x| and 2^-37 of the row's largest, in front of sum |w|."""
    w = synth.matrix(8, 2800 + cols, rows, cols)
    x = synth.activations_f32(2801 + tokens, (tokens, cols))
    x[0] *= np.float32(1e-20)
    x[-1] *= np.float32(1e4)
    check = np.unique(np.r_[0:200, np.linspace(0, rows - 1, 500).astype(int), rows // 2:rows // 2 + 40, rows - 40:rows])
    dense = orc.dequantize(8, np.ascontiguousarray(w.reshape(rows, -1)[check]).reshape(-1), len(check) * cols).reshape(len(check), cols).astype(np.float64)
    matrix, layout = (tsp.q8_lanes_pack_rows(cols, w), tsp.LAYOUT_Q8_LANES_V1) if lanes else (w, tsp.LAYOUT_GGUF)
    got = tsp.dense_mm_q8(gpu, layout, gpu.upload(matrix), gpu.upload(x), tokens, cols, rows).cpu().numpy()
    x64 = x.astype(np.float64)
    bound = (2.0 ** -18 + 2.0 ** -22) * (np.abs(x64) @ np.abs(dense).T) + 2.0 ** -37 * np.abs(x64).max(axis=1, keepdims=True) * np.abs(dense).sum(axis=1)
    assert gpu.error() == 0 and (np.abs(got[:, check] - x64 @ dense.T) <= bound).all()


# Token rows in registers, tile after tile: the sums have two places in turn, and the first is written again in a workgroup's third round (two tiles a round; one from
# nine waves on). Rounds of 131 072 matrix rows with one wave, 65 536 with two, 32 768 with three and four, 16 384 with five to eight, 8192 with nine and ten:
# into the second and into the third of each, the last round whole, of one tile, of one row, and with one tile of two
@pytest.mark.parametrize("lanes,tokens,cols,rows", [(False, 16, 256, 140001), (False, 9, 256, 270001), (False, 12, 512, 70001), (False, 9, 512, 131073), (False, 16, 768, 65600), (False, 8, 1024, 65600),
                                                    (False, 16, 1024, 100001), (False, 13, 1280, 40960), (False, 16, 1536, 32769), (False, 9, 1792, 41001), (False, 11, 2048, 49152),
                                                    (False, 16, 2048, 33001), (False, 7, 2304, 24576), (False, 12, 2560, 16417), (True, 12, 2560, 16417), (True, 16, 2560, 40001)])
def test_dense_mm_q8_resident_rounds(gpu, tsp, orc, synth, lanes, tokens, cols, rows):
    if cols > 2048:  # floats
        test_dense_mm_q8_f32_rows(gpu, tsp, orc, synth, lanes, tokens, cols, rows, 0)
    else:
        test_dense_mm_q8_halves_far_apart(gpu, tsp, orc, synth, lanes, tokens, cols, rows)


# a wave with whole matrix rows: one group of columns to eight, one item in flight and two, rounds of 2048 tiles with a last one of one row
@pytest.mark.parametrize("tokens,cols,rows", [(8, 256, 40001), (2, 256, 131073), (3, 1280, 72001), (1, 1280, 100000), (1, 1792, 52600), (8, 1792, 72033), (6, 1536, 65569), (4, 2048, 65537), (7, 2048, 131105),
                                              (8, 512, 65569), (8, 1024, 57345), (3, 2048, 57377), (5, 1536, 114721)])
def test_dense_mm_q8_rows_by_waves(gpu, tsp, orc, synth, tokens, cols, rows):
    """Some large matrices go to another kernel with up to eight token rows: the bits are those that the rows have in the company of others (twelve, which the
    other kernel takes), the bound that of the test above, and a value that is not finite is reported and spoils its own token's row alone."""
    w = synth.matrix(8, 2900 + cols, rows, cols)
    x = synth.activations_f32(2901 + tokens, (12, cols))
    x[0] *= np.float32(1e-20)
    x[tokens - 1, cols // 2:] *= np.float32(1e4)
    matrix = gpu.upload(w)
    few = lambda rows_of_x: tsp.dense_mm_q8(gpu, tsp.LAYOUT_GGUF, matrix, gpu.upload(rows_of_x), len(rows_of_x), cols, rows).cpu().numpy()
    got = few(x[:tokens])
    assert gpu.error() == 0
    assert np.array_equal(got.view(np.uint32), few(x)[:tokens].view(np.uint32)) and gpu.error() == 0
    check = np.unique(np.r_[0:200, rows // 2:rows // 2 + 40, rows - 40:rows])
    dense = orc.dequantize(8, np.ascontiguousarray(w.reshape(rows, -1)[check]).reshape(-1), len(check) * cols).reshape(len(check), cols).astype(np.float64)
    x64 = x[:tokens].astype(np.float64)
    bound = (2.0 ** -18 + 2.0 ** -22) * (np.abs(x64) @ np.abs(dense).T) + 2.0 ** -37 * np.abs(x64).max(axis=1, keepdims=True) * np.abs(dense).sum(axis=1)
    assert (np.abs(got[:, check] - x64 @ dense.T) <= bound).all()
    x[tokens - 1, cols - 1] = np.nan
    spoilt = few(x[:tokens])
    assert gpu.error() == tsp.ERRBIT_NONFINITE and np.array_equal(spoilt[:-1].view(np.uint32), got[:-1].view(np.uint32))


@pytest.mark.parametrize("lanes,tokens,cols,rows", [(False, 9, 512, 14003), (False, 16, 1024, 14002), (False, 7, 2560, 31001), (True, 13, 1024, 37), (True, 16, 2048, 515),
                                                    (True, 9, 2560, 1001), (False, 6, 2560, 33003), (False, 10, 2560, 22001)])
def test_dense_mm_q8_odd_rows(gpu, tsp, orc, synth, lanes, tokens, cols, rows):
    """An output that starts on any float and whose rows end on any: all of it is written and nothing around it, also where two workgroups to a matrix row add into
    one that was cleared before (2560 columns with six to ten token rows, q8_lanes_v1 rows with nine and more). Rows of two halves keep 22 bits of their
    largest value, and f32 sums 2^-18 of sum |w x|."""
    w = synth.matrix(8, 2700 + cols, rows, cols)
    x = synth.activations_f32(2701 + tokens, (tokens, cols))
    matrix = tsp.q8_lanes_pack_rows(cols, w) if lanes else w
    whole = gpu.full((tokens * rows + 8,), -5.0)
    for start in (1, 2, 4):
        whole.fill_(-5.0)
        out = whole[start:start + tokens * rows].view(tokens, rows)
        tsp.dense_mm_q8(gpu, tsp.LAYOUT_Q8_LANES_V1 if lanes else tsp.LAYOUT_GGUF, gpu.upload(matrix), gpu.upload(x), tokens, cols, rows, out=out)
        got = whole.cpu().numpy()
        assert (got[:start] == -5.0).all() and (got[start + tokens * rows:] == -5.0).all() and gpu.error() == 0
        got = got[start:start + tokens * rows].reshape(tokens, rows)
        check = np.unique(np.r_[0:min(rows, 200), max(0, rows - 40):rows])
        dense = orc.dequantize(8, np.ascontiguousarray(w.reshape(rows, -1)[check]).reshape(-1), len(check) * cols).reshape(len(check), cols).astype(np.float64)
        x64 = x.astype(np.float64)
        bound = 2.0 ** -18 * (np.abs(x64) @ np.abs(dense).T) + 2.0 ** -22 * np.abs(x64).max() * np.abs(dense).sum(axis=1)
        assert (np.abs(got[:, check] - x64 @ dense.T) <= bound).all()


@pytest.mark.parametrize("lanes,tokens,cols,rows", [(False, 9, 1024, 14003), (False, 16, 2048, 24576), (False, 10, 2560, 40001), (True, 13, 1024, 37), (True, 16, 2048, 512),
                                                    (True, 7, 2560, 1001), (True, 12, 2560, 64), (False, 6, 2560, 31003), (False, 9, 2560, 22001)])
def test_dense_mm_q8_sums_that_overflow_at_the_join(gpu, tsp, lanes, tokens, cols, rows):
    """Two workgroups to a matrix row (2560 columns with six to ten token rows, q8_lanes_v1 rows of up to 2048 with nine and more) or, the others, two waves to it, either
    half of whose sum is finite: a sum that passes the largest float is reported, wherever in the matrix it is, and halves of which one is nearly as
    large and the other takes it back are not."""
    blocks = np.zeros((rows, cols // 32, 34), dtype=np.uint8)
    blocks[:, :, 0:2] = np.array([4096.0], dtype=np.float16).view(np.uint8)
    blocks[:, 0, 2] = 1      # the first column and the last one
    blocks[:, -1, 33] = 1
    x = np.zeros((tokens, cols), dtype=np.float32)
    x[:, 0], x[:, -1] = 1.0 / 4096, 2.0 / 4096
    layout = tsp.LAYOUT_Q8_LANES_V1 if lanes else tsp.LAYOUT_GGUF

    def run(raw, token_rows):
        flat = np.ascontiguousarray(raw).reshape(-1)
        out = tsp.dense_mm_q8(gpu, layout, gpu.upload(tsp.q8_lanes_pack_rows(cols, flat) if lanes else flat), gpu.upload(token_rows), tokens, cols, rows)
        return gpu.error(), out.cpu().numpy()

    status, got = run(blocks, x)
    assert status == 0 and (got == 3.0).all()
    x[tokens - 1, 0], x[tokens - 1, -1] = 3.0 * 2.0 ** 114, -1.5 * 2.0 ** 114
    status, got = run(blocks, x)
    assert status == 0 and (got[tokens - 1] == np.float32(1.5 * 2.0 ** 126)).all()
    for row in (0, rows // 2, rows - 1):  # this row alone has the sum's second half with the sign turned round
        turned = blocks.copy()
        turned[row, -1, 33] = 255
        status, got = run(turned, x)
        assert np.isinf(got[tokens - 1, row]) and np.isfinite(np.delete(got, row, axis=1)).all()
        assert status == tsp.ERRBIT_NONFINITE
