"""GPU parity for the routed MoE over 1..8 token rows (decode / speculative verify), through the C
ABI, against the CPU composition dequantize -> double dot -> float SiLU -> double dot
(native/tests/test_planar_pack_v3.cpp:433-627; bound NMSE <= 1e-6)."""
import importlib

import numpy as np
import pytest

from conftest import max_rel_error, nmse, reference_metric

pytestmark = pytest.mark.gpu


def lcg_inputs(seed, count):
    # native/tests/test_planar_pack_v3.cpp:489-494
    out = np.empty(count, dtype=np.float32)
    rng = seed
    for i in range(count):
        rng = (rng * 1664525 + 1013904223) & 0xFFFFFFFF
        out[i] = np.float32(int(rng % 1993) - 996) / np.float32(997.0)
    return out


def build(tsp, gpu, orc, gu, dn, channels, hidden, experts, distinct_up=True):
    gate = orc.fixture_weights(gu, channels, hidden, experts)
    up = gate.copy()
    if distinct_up:  # the reference fixture reuses one generator; flip quant bytes so gate != up
        bpb = orc.encoding(gu)[1]
        keep = 16 if gu == 12 else 48 if gu == 13 else 2
        blocks = up.reshape(-1, bpb)
        blocks[:, keep:] ^= 0x5A
    if dn == 14:  # the LCG fixture fixes the f16 scale at byte 0; Q6_K keeps it at byte 208, so draw valid blocks instead
        down = importlib.import_module("tokspur-public_amd.synth").matrix(14, 4242, channels * experts, hidden)
    else:
        down = orc.fixture_weights(dn, hidden, channels, experts)
    return gate, up, down, tsp.PlanarMoeWeights(gpu, gu, dn, channels, hidden, experts, gate, up, down)


@pytest.mark.parametrize("gu,dn", [(12, 7), (13, 7), (13, 8), (8, 8), (12, 14)])
def test_routed_m8_reference_cases(gpu, tsp, orc, gu, dn):
    # native/tests/test_planar_pack_v3.cpp:440-551: every width 1..8 with shared experts (0 and 5) and singletons.
    channels, hidden, experts, selected = (256, 64, 8, 4) if dn != 14 else (256, 256, 8, 4)
    gate, up, down, w = build(tsp, gpu, orc, gu, dn, channels, hidden, experts)
    for m in range(1, 9):
        x = lcg_inputs(9001 + m * 31 + gu, m * channels).reshape(m, channels)
        ids = np.array([[0 if s == 0 else 5 if (s == 1 and t & 1) else (t * 3 + s * 2 + 1) % experts for s in range(selected)]
                        for t in range(m)], dtype=np.uint32).reshape(-1)
        h, y = tsp.planar_moe_routed_m8(gpu, w, gpu.upload(ids), gpu.upload(x), m, selected)
        ref_h, ref_y = orc.moe_routed_reference(gu, dn, gate, up, down, channels, hidden, experts, ids, m, selected, x, threads=4)
        assert nmse(h.cpu().numpy(), ref_h) <= 1e-6 and nmse(y.cpu().numpy(), ref_y) <= 1e-6, m
        assert gpu.error() == 0
        only_h = tsp.planar_moe_gate_up_swiglu_m8(gpu, w, gpu.upload(ids), gpu.upload(x), m, selected)
        assert np.array_equal(only_h.cpu().numpy(), h.cpu().numpy())


@pytest.mark.parametrize("dn,hidden", [(7, 160), (8, 96)])
@pytest.mark.parametrize("tokens", [2, 5, 8])
def test_routed_m8_2048_columns_narrow_experts(gpu, tsp, orc, dn, hidden, tokens):
    """Experts of 2048 columns whose hidden width is no multiple of 128 (five and three 32-unit tiles) on the kernel that keeps
    the step's token rows resident: the share split by 32-unit tiles and the hand-off to a Q5_1 / Q8_0 down product."""
    channels, experts, selected = 2048, 8, 3
    gate, up, down, w = build(tsp, gpu, orc, 12, dn, channels, hidden, experts)
    x = lcg_inputs(555 + tokens * 17 + hidden, tokens * channels).reshape(tokens, channels)
    ids = np.array([[(t * 2 + s * 3) % experts for s in range(selected)] for t in range(tokens)], dtype=np.uint32).reshape(-1)
    h, y = tsp.planar_moe_routed_m8(gpu, w, gpu.upload(ids), gpu.upload(x), tokens, selected)
    ref_h, ref_y = orc.moe_routed_reference(12, dn, gate, up, down, channels, hidden, experts, ids, tokens, selected, x, threads=4)
    assert nmse(h.cpu().numpy(), ref_h) <= 1e-6 and nmse(y.cpu().numpy(), ref_y) <= 1e-6
    assert gpu.error() == 0


@pytest.mark.parametrize("gu,dn", [(12, 7), (8, 8)])
def test_routed_m8_all_singletons(gpu, tsp, orc, gu, dn):
    # native/tests/test_planar_pack_v3.cpp:553-627: 32 experts, every route a distinct expert, hidden = 416 (13 blocks).
    channels, hidden, experts, selected = 512, 416, 32, 4
    gate, up, down, w = build(tsp, gpu, orc, gu, dn, channels, hidden, experts)
    for m in range(2, 9):
        x = lcg_inputs(31337 + m * 23 + gu * 7, m * channels).reshape(m, channels)
        ids = np.array([(rid * 7 + 3) % experts for rid in range(m * selected)], dtype=np.uint32)
        h, y = tsp.planar_moe_routed_m8(gpu, w, gpu.upload(ids), gpu.upload(x), m, selected)
        ref_h, ref_y = orc.moe_routed_reference(gu, dn, gate, up, down, channels, hidden, experts, ids, m, selected, x, threads=4)
        assert nmse(h.cpu().numpy(), ref_h) <= 1e-6 and nmse(y.cpu().numpy(), ref_y) <= 1e-6, m
    assert gpu.error() == 0


# rows of 1, 2, 4, 8 super-blocks take the one-block-per-wave kernel, (768, 1280) the looped one on both sides
@pytest.mark.parametrize("channels,hidden", [(2048, 512), (1024, 256), (512, 1024), (256, 2048), (768, 1280)])
@pytest.mark.parametrize("tokens", [1, 2, 3, 5, 8])
def test_routed_m8_fast_arms(gpu, tsp, orc, synth, channels, hidden, tokens):
    """Q4_K co-located gate/up with Q6_K planes for down: the shapes the register-resident kernels take,
    with repeated experts (records of several tokens), strided rows and canary padding."""
    experts, selected = 8, 4
    gate = synth.matrix(12, 21, hidden * experts, channels)
    up = synth.matrix(12, 22, hidden * experts, channels)
    down = synth.matrix(14, 23, channels * experts, hidden)
    w = tsp.PlanarMoeWeights(gpu, 12, 14, channels, hidden, experts, gate, up, down)
    rng = np.random.default_rng(tokens)
    others = [e for e in range(experts) if e != 3]  # expert 3 is shared by every token
    ids = np.array([[3] + list(rng.permutation(others)[:selected - 1]) for _ in range(tokens)], dtype=np.uint32).reshape(-1)
    x = (synth.activations_f32(24 + tokens, (tokens, channels + 16)) * 0.1).astype(np.float32)
    routes = tokens * selected
    h = gpu.full((routes, hidden + 4), -5.0)
    y = gpu.full((routes, channels + 8), -6.0)
    tsp.planar_moe_routed_m8(gpu, w, gpu.upload(ids), gpu.upload(x), tokens, selected, h=h, y=y,
                             x_stride=(channels + 16) * 4, h_stride=(hidden + 4) * 4, y_stride=(channels + 8) * 4)
    ref_h, ref_y = orc.moe_routed_reference(12, 14, gate, up, down, channels, hidden, experts, ids, tokens, selected,
                                            np.ascontiguousarray(x[:, :channels]), threads=8)
    h, y = h.cpu().numpy(), y.cpu().numpy()
    assert nmse(h[:, :hidden], ref_h) <= 1e-6 and nmse(y[:, :channels], ref_y) <= 1e-6
    assert (h[:, hidden:] == -5.0).all() and (y[:, channels:] == -6.0).all() and gpu.error() == 0


@pytest.mark.parametrize("channels,hidden", [(2048, 512), (512, 256), (768, 1280)])
@pytest.mark.parametrize("tokens", [1, 3, 8])
def test_routed_m8_with_always_on_expert(gpu, tsp, orc, synth, channels, hidden, tokens):
    """The layer's always-on expert as one more record of the two launches (its rows are the tokens): the routed rows are
    the same bits as without it, its rows the same bits as a separate call that routes every token to it, and they agree
    with the CPU composition; padding of a strided output stays."""
    experts, selected = 8, 3
    gate = synth.matrix(12, 41, hidden * experts, channels)
    up = synth.matrix(12, 42, hidden * experts, channels)
    down = synth.matrix(14, 43, channels * experts, hidden)
    sg, su, sd = synth.matrix(12, 44, hidden, channels), synth.matrix(12, 45, hidden, channels), synth.matrix(14, 46, channels, hidden)
    w = tsp.PlanarMoeWeights(gpu, 12, 14, channels, hidden, experts, gate, up, down)
    shared = tsp.PlanarSharedExpert(gpu, channels, hidden, sg, su, sd)
    rng = np.random.default_rng(tokens + channels)
    ids = np.stack([rng.permutation(experts)[:selected] for _ in range(tokens)]).astype(np.uint32).reshape(-1)
    x = (synth.activations_f32(47 + tokens, (tokens, channels)) * 0.25).astype(np.float32)
    d_ids, d_x = gpu.upload(ids), gpu.upload(x)
    h0, y0 = tsp.planar_moe_routed_m8(gpu, w, d_ids, d_x, tokens, selected)
    padded = gpu.full((tokens, channels + 4), -2.0)
    h1, y1, _ = tsp.planar_moe_routed_m8(gpu, w, d_ids, d_x, tokens, selected, shared=shared, shared_y=padded, shared_y_stride=(channels + 4) * 4)
    assert gpu.error() == 0
    assert np.array_equal(h1.cpu().numpy().view(np.uint32), h0.cpu().numpy().view(np.uint32))
    assert np.array_equal(y1.cpu().numpy().view(np.uint32), y0.cpu().numpy().view(np.uint32))
    got = padded.cpu().numpy()
    assert (got[:, channels:] == -2.0).all()
    alone = tsp.PlanarMoeWeights(gpu, 12, 14, channels, hidden, 2, np.concatenate([sg, sg]), np.concatenate([su, su]), np.concatenate([sd, sd]))
    zeros = np.zeros(tokens, dtype=np.uint32)
    _, separate = tsp.planar_moe_routed_m8(gpu, alone, gpu.upload(zeros), d_x, tokens, 1)
    assert np.array_equal(got[:, :channels].view(np.uint32), separate.cpu().numpy().view(np.uint32))
    _, ref_y = orc.moe_routed_reference(12, 14, sg, su, sd, channels, hidden, 1, zeros, tokens, 1, x, threads=4)
    assert nmse(got[:, :channels], ref_y) <= 1e-6
    other = tsp.PlanarMoeWeights(gpu, 13, 7, 256, 256, 2, synth.matrix(13, 1, 512, 256), synth.matrix(13, 2, 512, 256), synth.matrix(7, 3, 512, 256))
    small = tsp.PlanarSharedExpert(gpu, 256, 256, synth.matrix(12, 4, 256, 256), synth.matrix(12, 5, 256, 256), synth.matrix(14, 6, 256, 256))
    with pytest.raises(tsp.FormatError):  # only beside the Q4_K / Q6_K kinds
        tsp.planar_moe_routed_m8(gpu, other, gpu.upload(np.zeros(2, dtype=np.uint32)), gpu.zeros((2, 256)), 2, 1, shared=small)


def test_routed_m8_sticky_errors_and_refusals(gpu, tsp, orc, synth):
    channels, hidden, experts, selected = 512, 256, 4, 2
    gate = synth.matrix(12, 31, hidden * experts, channels)
    down = synth.matrix(14, 33, channels * experts, hidden)
    w = tsp.PlanarMoeWeights(gpu, 12, 14, channels, hidden, experts, gate, gate, down)
    x = synth.activations_f32(34, (2, channels))
    good = gpu.upload(np.array([0, 1, 2, 3], dtype=np.uint32))
    tsp.planar_moe_routed_m8(gpu, w, gpu.upload(np.array([0, 1, 2, 4], dtype=np.uint32)), gpu.upload(x), 2, selected)
    assert gpu.error() & tsp.ERRBIT_INDEX
    bad = x.copy()
    bad[1, 5] = np.inf
    tsp.planar_moe_routed_m8(gpu, w, good, gpu.upload(bad), 2, selected)
    assert gpu.error() & tsp.ERRBIT_NONFINITE
    h, y = tsp.planar_moe_routed_m8(gpu, w, good, gpu.upload(x), 2, selected)  # the next batch is clean
    assert gpu.error() == 0 and np.isfinite(y.cpu().numpy()).all()
    # the same through the launch that keeps the tokens resident and builds the union records itself (2048-column experts)
    wide = tsp.PlanarMoeWeights(gpu, 12, 14, 2048, 256, experts, synth.matrix(12, 35, 256 * experts, 2048), synth.matrix(12, 36, 256 * experts, 2048),
                                synth.matrix(14, 37, 2048 * experts, 256))
    xw = synth.activations_f32(38, (2, 2048))
    h, y = tsp.planar_moe_routed_m8(gpu, wide, good, gpu.upload(xw), 2, selected)
    assert gpu.error() == 0 and np.isfinite(y.cpu().numpy()).all()
    before = y.cpu().numpy().copy()
    tsp.planar_moe_routed_m8(gpu, wide, gpu.upload(np.array([0, 1, 7, 3], dtype=np.uint32)), gpu.upload(xw), 2, selected, y=y)
    assert gpu.error() & tsp.ERRBIT_INDEX and np.array_equal(y.cpu().numpy(), before)  # nothing ran on the bad batch
    h, y2 = tsp.planar_moe_routed_m8(gpu, wide, good, gpu.upload(xw), 2, selected)
    assert gpu.error() == 0 and np.array_equal(y2.cpu().numpy(), before)
    with pytest.raises(tsp.FormatError):
        tsp.planar_moe_routed_m8(gpu, w, good, gpu.upload(x), 9, selected)
    with pytest.raises(tsp.FormatError):
        tsp.planar_moe_routed_m8(gpu, w, good, gpu.upload(x), 2, 17)
    with pytest.raises(tsp.FormatError):  # output aliasing the activations
        xd = gpu.upload(np.zeros((4, channels), dtype=np.float32))
        tsp.planar_moe_routed_m8(gpu, w, good, xd, 2, selected, y=xd)


def test_routed_m8_through_ctypes(gpu, tsp, orc):
    """A program that binds the C ABI with ctypes and the exported structures gets the compiled binding's bits."""
    import ctypes
    channels, hidden, experts, selected, tokens = 256, 64, 8, 4, 3
    w = build(tsp, gpu, orc, 12, 7, channels, hidden, experts)[3]
    ids = gpu.upload(np.array([[0, 3, 5, 7], [1, 0, 2, 4], [6, 5, 0, 1]], dtype=np.uint32).reshape(-1))
    x = gpu.upload(lcg_inputs(77, tokens * channels).reshape(tokens, channels))
    h, y = tsp.planar_moe_routed_m8(gpu, w, ids, x, tokens, selected)
    h2, y2 = gpu.zeros(h.shape), gpu.zeros(y.shape)
    m = tsp.SmallMoe(w.pair_lo.data_ptr(), w.pair_hi.data_ptr(), w.down.data_ptr(), *tsp.COLOC_KINDS[12], tsp.DOWN_KINDS[7], channels, hidden, experts, selected,
                     tokens, ids.data_ptr(), x.data_ptr(), channels * 4, h2.data_ptr(), hidden * 4, y2.data_ptr(), channels * 4, w.union_meta.data_ptr(),
                     gpu.err.data_ptr())
    assert tsp.dll().tsp_planar_moe_routed_m8(ctypes.byref(m), gpu.stream()) == tsp.OK and gpu.error() == 0
    assert np.array_equal(h2.cpu().numpy(), h.cpu().numpy()) and np.array_equal(y2.cpu().numpy(), y.cpu().numpy())


def test_config2_moe_verify(gpu, tsp, orc, synth):
    """BASELINE config 2 at full size: T = 8, hidden 2048, 512 experts, top-10 renormalised softmax routing,
    gate+up Q4_K [2x512, 2048], down Q6_K [2048, 512]; router -> routed experts -> weighted combine with an
    always-on shared expert (shared_logit = 20, so sigmoid(shared_logit) rounds to 1 in f32)."""
    T, C, H, E, S = 8, 2048, 512, 512, 10
    logits = synth.activations_f32(synth.tensor_seed(2, 1), (T, E))
    x = synth.activations_f32(synth.tensor_seed(2, 2), (T, C))
    ids_d, wts_d = gpu.route(gpu.upload(logits), S, 0, True, tokens=T)
    ids = ids_d.cpu().numpy().view(np.uint32).reshape(-1)
    want_ids = np.concatenate([orc.route_reference(logits[t].astype(np.float64), S, 0, True)[0] for t in range(T)])
    assert np.array_equal(ids, want_ids)
    used = sorted(set(int(e) for e in ids))
    gu_spec, dn_spec = tsp.make_expert_spec(12, C, H), tsp.make_expert_spec(14, H, C)
    # only the experts the routes touch are materialised; the rest of the 1 GB tensors stay zero and are never read
    w = object.__new__(tsp.PlanarMoeWeights)
    w.gu_type, w.dn_type, w.channels, w.hidden, w.experts, w.gu_spec, w.dn_spec = 12, 14, C, H, E, gu_spec, dn_spec
    pb, db = gu_spec.planar_expert_bytes, dn_spec.planar_expert_bytes
    w.pair_lo, w.pair_hi = gpu.zeros(E // 2 * 2 * pb, "uint8"), gpu.zeros(E // 2 * 2 * pb, "uint8")
    w.down, w.union_meta = gpu.zeros(E * db, "uint8"), gpu.zeros(2320, "int32")
    raw = {}
    for e in used:
        g = synth.matrix(12, synth.tensor_seed(2, 1000 + e), H, C)
        u = synth.matrix(12, synth.tensor_seed(2, 2000 + e), H, C)
        d = synth.matrix(14, synth.tensor_seed(2, 3000 + e), C, H)
        raw[e] = (g, u, d)
        half, local = (w.pair_lo, e) if e < E // 2 else (w.pair_hi, e - E // 2)
        half[local * 2 * pb:local * 2 * pb + pb] = gpu.upload(tsp.pack_expert(gu_spec, g))
        half[local * 2 * pb + pb:(local + 1) * 2 * pb] = gpu.upload(tsp.pack_expert(gu_spec, u))
        w.down[e * db:(e + 1) * db] = gpu.upload(tsp.pack_expert(dn_spec, d))
    h, y = tsp.planar_moe_routed_m8(gpu, w, ids_d, gpu.upload(x), T, S)
    # shared expert: the same shapes, dense (one "route" per token through a 2-expert stack whose expert 0 is used)
    sg = synth.matrix(12, synth.tensor_seed(2, 10), H, C)
    su = synth.matrix(12, synth.tensor_seed(2, 11), H, C)
    sd = synth.matrix(14, synth.tensor_seed(2, 12), C, H)
    ws = tsp.PlanarMoeWeights(gpu, 12, 14, C, H, 2, np.concatenate([sg, sg]), np.concatenate([su, su]), np.concatenate([sd, sd]))
    _, ys = tsp.planar_moe_routed_m8(gpu, ws, gpu.zeros(T, "int32"), gpu.upload(x), T, 1)
    out = gpu.mixture(y, wts_d, ys, gpu.full(T, 20.0), C, S, tokens=T).cpu().numpy()
    assert gpu.error() == 0
    # the same step as the bench runs it: the shared expert as one more record of the routed experts' two launches
    riding = tsp.PlanarSharedExpert(gpu, C, H, sg, su, sd)
    h2, y2, ys2 = tsp.planar_moe_routed_m8(gpu, w, ids_d, gpu.upload(x), T, S, shared=riding)
    assert gpu.error() == 0
    assert np.array_equal(y2.cpu().numpy().view(np.uint32), y.cpu().numpy().view(np.uint32))
    assert np.array_equal(ys2.cpu().numpy().view(np.uint32), ys.cpu().numpy().view(np.uint32))

    # oracle: per-route experts through compact stacks (expert index = position in `used`)
    pos = {e: i for i, e in enumerate(used)}
    cg = np.concatenate([raw[e][0] for e in used]); cu = np.concatenate([raw[e][1] for e in used]); cd = np.concatenate([raw[e][2] for e in used])
    cid = np.array([pos[int(e)] for e in ids], dtype=np.uint32)
    ref_h, ref_y = orc.moe_routed_reference(12, 14, cg, cu, cd, C, H, len(used), cid, T, S, x, threads=8)
    _, ref_ys = orc.moe_routed_reference(12, 14, sg, su, sd, C, H, 1, np.zeros(T, dtype=np.uint32), T, 1, x, threads=8)
    assert nmse(h.cpu().numpy(), ref_h) <= 1e-6 and nmse(y.cpu().numpy(), ref_y) <= 1e-6
    want = np.stack([orc.mixture_reference(ref_y[t * S:(t + 1) * S], orc.route_reference(logits[t].astype(np.float64), S, 0, True)[1],
                                           ref_ys[t], 20.0) for t in range(T)])
    # Outputs here are ~1e6 in magnitude (weights up to ~19 and ~60, two stacked projections), so the bar is the
    # engine's MoE bound (NMSE <= 1e-6) plus max error <= 2e-3 in units of each row's scale.
    print(f"config2: {len(used)} distinct experts, NMSE {nmse(out, want):.3e}, max rel error {max_rel_error(out, want):.3e}")
    assert nmse(out, want) <= 1e-6 and max_rel_error(out, want) <= 2e-3
    # the engine's own metric for the record (outputs of magnitude ~1e6: see reference_metric)
    value, at, actual, expected, row_rms = reference_metric(out, want)
    print(f"config2: reference metric |a-e|/max(1,|e|) = {value:.3e} at element {at} (got {actual:.8g}, reference {expected:.8g}, "
          f"row rms {row_rms:.3g}: {abs(actual - expected) / row_rms:.2e} of the row scale)")


@pytest.mark.parametrize("tokens", [1, 2, 5, 8])
@pytest.mark.parametrize("dn,channels,hidden,experts,selected", [(8, 2560, 640, 16, 10), (7, 2560, 160, 8, 4), (14, 1280, 768, 8, 4), (8, 256, 32, 4, 2),
                                                                 (7, 768, 2560, 4, 2), (8, 1792, 96, 64, 16)])
def test_routed_m8_streamed(gpu, tsp, orc, synth, dn, channels, hidden, experts, selected, tokens):
    """The streaming kernels: rows of 1 to 10 super-blocks, down rows that do not fill their last 128 columns (160, 96, 32), more
    rows than one pass holds (every token on expert 0), shares that span several records, strided rows and canaries; a row's
    bits do not depend on which tokens ride along."""
    gate, up = synth.matrix(12, 51, hidden * experts, channels), synth.matrix(12, 52, hidden * experts, channels)
    down = synth.matrix(dn, 53, channels * experts, hidden)
    w = tsp.PlanarMoeWeights(gpu, 12, dn, channels, hidden, experts, gate, up, down)
    rng = np.random.default_rng(tokens + channels)
    ids = np.array([[0] + list(1 + rng.permutation(experts - 1)[:selected - 1]) for _ in range(tokens)], dtype=np.uint32)
    x = (synth.activations_f32(54 + tokens, (tokens, channels + 8)) * 0.1).astype(np.float32)
    routes = tokens * selected
    h, y = gpu.full((routes, hidden + 4), -5.0), gpu.full((routes, channels + 8), -6.0)
    tsp.planar_moe_routed_m8(gpu, w, gpu.upload(ids.reshape(-1)), gpu.upload(x), tokens, selected, h=h, y=y, x_stride=(channels + 8) * 4,
                             h_stride=(hidden + 4) * 4, y_stride=(channels + 8) * 4)
    h, y = h.cpu().numpy(), y.cpu().numpy()
    ref_h, ref_y = orc.moe_routed_reference(12, dn, gate, up, down, channels, hidden, experts, ids.reshape(-1), tokens, selected,
                                            np.ascontiguousarray(x[:, :channels]), stage=8 if dn == 14 else 0, threads=8)
    # a row of two halves has 22 bits of its largest value, 2^-22 of the row or 6e-14 here; one half alone is 4e-8. (Stage bit 8: a Q6_K
    # product sc * (q - 32) above 2048 loses its lowest bit as a half, which is 1.8e-8 against the exact weights.)
    assert nmse(h[:, :hidden], ref_h) <= 1e-12 and nmse(y[:, :channels], ref_y) <= 1e-12
    assert (h[:, hidden:] == -5.0).all() and (y[:, channels:] == -6.0).all() and gpu.error() == 0
    if tokens > 2:  # two or more tokens take the same kernels
        _, pair = tsp.planar_moe_routed_m8(gpu, w, gpu.upload(ids[-2:].reshape(-1)), gpu.upload(np.ascontiguousarray(x[-2:, :channels])), 2, selected)
        assert np.array_equal(pair.cpu().numpy().view(np.uint32), np.ascontiguousarray(y[-2 * selected:, :channels]).view(np.uint32))


@pytest.mark.parametrize("tokens", [1, 4, 5, 6, 8])
@pytest.mark.parametrize("dn,channels,hidden", [(8, 2560, 640), (7, 2304, 160), (8, 1280, 96), (7, 768, 2560), (14, 256, 2304)])
def test_routed_m8_streamed_f32(gpu, tsp, orc, synth, dn, channels, hidden, tokens):
    """Rows of more than 2048 columns, and all rows of Q8_0 and Q5_1, are multiplied as the floats they are, also
    where every token meets one expert (more rows than one pass has room for): values 1e6 to 1e30 beside ordinary ones, in front
    of weights that are zero, take nothing from them.
    Error bound: eight roundings of a block's sums and one for each of at most 80 blocks, of the sum of |scale * code| + |minimum|
    times |x|, less than 2^-17 of it; the expected values take the rows that the device itself has."""
    experts, selected = 8, 2
    gate, up = synth.matrix(12, 61, hidden * experts, channels), synth.matrix(12, 62, hidden * experts, channels)
    down = synth.matrix(dn, 63, channels * experts, hidden)
    for raw in (gate, up):  # weight 5 of every 256: a sub-block without minimum, the code zero
        blocks = raw.reshape(-1, 144)
        blocks[:, 8] &= 0xC0
        blocks[:, 16 + 5] &= 0xF0
    # hidden units 5, 101, 197, ... come out some 2^26 times the others
    for raw, factor in ((gate, 2.0 ** 6), (up, 2.0 ** 20)):
        scales = raw.reshape(experts, hidden, channels // 256, 144)[:, 5::96, :, 0:4]
        scales[:] = np.minimum(np.ascontiguousarray(scales).view(np.float16).astype(np.float64) * factor, 60000).astype(np.float16).view(np.uint8)
    blocks = down.reshape(-1, 210) if dn == 14 else down.reshape(experts * channels, hidden // 32, -1)[:, ::3]
    if dn == 14:
        blocks[:, [5, 37, 69, 101]] = 0
        blocks[:, [133, 165]] = 0xaa
    elif dn == 8:
        blocks[:, :, 2 + 5] = 0
    else:
        blocks[:, :, 2:4] = 0
        blocks[:, :, 4] &= 0xDF  # the fifth bit
        blocks[:, :, 8 + 5] &= 0xF0
    w = tsp.PlanarMoeWeights(gpu, 12, dn, channels, hidden, experts, gate, up, down)
    ids = np.array([[3, (t + 4) % experts] if t != 2 else [3, 1] for t in range(tokens)], dtype=np.uint32).reshape(-1)
    x = (synth.activations_f32(64 + tokens, (tokens, channels)) * 0.1).astype(np.float32)
    if channels > 2048:  # up to there a row is two halves under one scale
        x[:, 5::256] = np.resize(np.array([1e6, -3e12, 1e30], dtype=np.float32), channels // 256)
    x[tokens // 2] *= np.float32(1e-12)
    h, y = tsp.planar_moe_routed_m8(gpu, w, gpu.upload(ids), gpu.upload(x), tokens, selected)
    h, y = h.cpu().numpy().astype(np.float64), y.cpu().numpy().astype(np.float64)
    assert gpu.error() == 0

    def weights(t, raw, rows, cols):  # the weights of each expert, and |scale * code| + |minimum|
        value = orc.dequantize(t, raw, experts * rows * cols).astype(np.float64).reshape(experts, rows, cols)
        if t in (8, 14):
            return value, np.abs(value)
        least = raw.copy()
        b = least.reshape(-1, 144 if t == 12 else 24)
        b[:, 0:2] = 0  # no scale: the minima alone
        least = np.abs(orc.dequantize(t, least, value.size).astype(np.float64).reshape(value.shape))
        return value, np.abs(value) + 2 * least

    (gate_w, gate_a), (up_w, up_a), (down_w, down_a) = weights(12, gate, hidden, channels), weights(12, up, hidden, channels), weights(dn, down, channels, hidden)
    unit = 2.0 ** -17
    for r, e in enumerate(ids):
        row = x[r // selected].astype(np.float64)
        g, u, dg, du = gate_w[e] @ row, up_w[e] @ row, unit * (gate_a[e] @ np.abs(row)), unit * (up_a[e] @ np.abs(row))
        s = 1 / (1 + np.exp(-np.clip(g, -700, 700)))
        bound = 1.1 * dg * (np.abs(u) + du) + np.abs(g * s) * du + 2.0 ** -20 * np.abs(g * s * u) + 1e-36
        assert (np.abs(h[r] - g * s * u) <= bound).all(), (r, float(np.max(np.abs(h[r] - g * s * u) / bound)))
        bound = unit * (down_a[e] @ np.abs(h[r])) + 1e-36
        assert (np.abs(y[r] - down_w[e] @ h[r]) <= bound).all(), (r, float(np.max(np.abs(y[r] - down_w[e] @ h[r]) / bound)))


@pytest.mark.parametrize("tokens", [1, 3, 7])
@pytest.mark.parametrize("dn,channels,hidden", [(8, 2560, 96), (7, 2304, 160), (14, 1280, 768), (8, 768, 640)])
def test_routed_m8_streamed_errors(gpu, tsp, synth, dn, channels, hidden, tokens):
    """The streaming kernels: a value that is not finite in a row, an infinite scale in a block of the down weights and an expert id
    out of range are reported, the rows of other weights and experts keep their bits (also the row before the infinite block, where a
    step of 128 columns reads across), and the next batch is clean."""
    experts, selected = 6, 2
    gate, up = synth.matrix(12, 71, hidden * experts, channels), synth.matrix(12, 72, hidden * experts, channels)
    w = tsp.PlanarMoeWeights(gpu, 12, dn, channels, hidden, experts, gate, up, synth.matrix(dn, 73, channels * experts, hidden))
    ids = np.array([[2, t % 2 * 3 + 1] for t in range(tokens)], dtype=np.uint32).reshape(-1)
    x = (synth.activations_f32(74, (tokens, channels)) * 0.1).astype(np.float32)
    good_ids, good_x, routes = gpu.upload(ids), gpu.upload(x), tokens * selected

    def run(d_ids, d_x):
        h, y = gpu.full((routes, hidden), -3.0), gpu.full((routes, channels), -4.0)
        tsp.planar_moe_routed_m8(gpu, w, d_ids, d_x, tokens, selected, h=h, y=y)
        return gpu.error(), y.cpu().numpy()

    status, want = run(good_ids, good_x)
    assert status == 0 and np.isfinite(want).all()
    for value in (np.inf, np.nan):
        bad = x.copy()
        bad[tokens - 1, channels - 1] = value
        status, y = run(good_ids, gpu.upload(bad))
        assert status == tsp.ERRBIT_NONFINITE and np.array_equal(y[:routes - selected], want[:routes - selected])
    size, row, expert = (4 if dn == 7 else 2), 17, 2
    at = expert * w.dn_spec.planar_expert_bytes + w.dn_spec.dm_offset + row * w.dn_spec.blocks_per_row * size
    kept = w.down[at:at + 2].clone()
    w.down[at:at + 2] = gpu.upload(np.array([0x00, 0x7C], dtype=np.uint8))
    status, y = run(good_ids, good_x)
    w.down[at:at + 2] = kept
    assert status == tsp.ERRBIT_NONFINITE and not np.isfinite(y[ids == expert, row]).any()
    y[ids == expert, row] = want[ids == expert, row]
    assert np.array_equal(y, want)
    poisoned = ids.copy()
    poisoned[routes - 1] = experts
    status, y = run(gpu.upload(poisoned), good_x)
    assert status == tsp.ERRBIT_INDEX
    if tokens > 1:
        assert (y == -4.0).all()  # no record of the batch stands
    else:
        assert np.array_equal(y[0], want[0]) and (y[1] == -4.0).all()
    status, y = run(good_ids, good_x)
    assert status == 0 and np.array_equal(y, want)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dn,channels,hidden", [(14, 3072, 1024), (14, 1024, 512), (14, 2048, 768), (14, 512, 256), (8, 2048, 1024), (8, 2304, 544),
                                                (7, 1280, 736), (7, 1024, 992), (7, 256, 512)])
def test_routed_m8_one_token(gpu, tsp, orc, synth, dn, channels, hidden, offset):
    """One token: every split of a row over lanes and units, full and with a tail, the widest rows these kernels take, a token row and
    route rows that only floats align (offset 1). Sums of f32 products: a rounding or two of 2^-24 per value and partial sum, an
    error of less than 2^-20 of the row's size, 1e-12 of its square. (Stage bit 8: a Q6_K product sc * (q - 32) is a half, of route rows that
    16 bytes align; of others every weight is the float that it decodes to.)"""
    experts, selected = 6, 4
    gate, up = synth.matrix(12, 91, hidden * experts, channels), synth.matrix(12, 92, hidden * experts, channels)
    down = synth.matrix(dn, 93, channels * experts, hidden)
    w = tsp.PlanarMoeWeights(gpu, 12, dn, channels, hidden, experts, gate, up, down)
    ids = np.array([5, 0, 3, 2], dtype=np.uint32)
    x = (synth.activations_f32(94, (1, channels)) * 0.1).astype(np.float32)
    d_x = gpu.upload(np.concatenate([np.zeros((1, offset), dtype=np.float32), x], axis=1))[:, offset:]
    h, y = gpu.full((selected, hidden + 4 + offset), -5.0), gpu.full((selected, channels + 4), -6.0)
    tsp.planar_moe_routed_m8(gpu, w, gpu.upload(ids), d_x, 1, selected, h=h, y=y, x_stride=(channels + offset) * 4,
                             h_stride=(hidden + 4 + offset) * 4, y_stride=(channels + 4) * 4)
    h, y = h.cpu().numpy(), y.cpu().numpy()
    ref_h, ref_y = orc.moe_routed_reference(12, dn, gate, up, down, channels, hidden, experts, ids, 1, selected, x, stage=8 if dn == 14 and offset == 0 else 0, threads=8)
    assert nmse(h[:, :hidden], ref_h) <= 1e-12 and nmse(y[:, :channels], ref_y) <= 1e-12
    assert (h[:, hidden:] == -5.0).all() and (y[:, channels:] == -6.0).all() and gpu.error() == 0


@pytest.mark.parametrize("dn,channels,hidden,experts,selected,tokens", [(8, 256, 1280, 20, 16, 8), (14, 512, 1280, 6, 6, 5), (7, 3328, 96, 4, 1, 3),
                                                                        (14, 2048, 512, 64, 10, 8), (8, 3328, 640, 8, 2, 1), (7, 512, 1056, 8, 3, 2)])
def test_routed_m8_few_tokens(gpu, tsp, orc, synth, dn, channels, hidden, experts, selected, tokens):
    """Experts met by one, two and many tokens, routes on both sides of the sixty-fourth, a token with the same expert twice, the splits of
    wide rows over lanes, rows that only floats align; and the union block that the call leaves for its caller. A row's bits don't depend on
    the tokens beside it. Sums of f32 products: see the test of one token. (Q6_K down rows: a second call with route rows that 16 bytes align.)"""
    gate, up = synth.matrix(12, 95, hidden * experts, channels), synth.matrix(12, 96, hidden * experts, channels)
    down = synth.matrix(dn, 97, channels * experts, hidden)
    w = tsp.PlanarMoeWeights(gpu, 12, dn, channels, hidden, experts, gate, up, down)
    rng = np.random.default_rng(channels + tokens)
    ids = np.stack([rng.permutation(experts)[:selected] for _ in range(tokens)]).astype(np.uint32)
    ids[0, -1] = ids[0, 0]
    x = (synth.activations_f32(98, (tokens, channels + 1)) * 0.1).astype(np.float32)
    routes = tokens * selected
    w.union_meta.fill_(-1)

    def run(rows, x_rows, pad=1):
        h, y = gpu.full((rows.size, hidden + pad), -5.0), gpu.full((rows.size, channels + 4), -6.0)
        tsp.planar_moe_routed_m8(gpu, w, gpu.upload(rows.reshape(-1)), gpu.upload(x_rows)[:, 1:], len(rows), selected, h=h, y=y, x_stride=(channels + 1) * 4,
                                 h_stride=(hidden + pad) * 4, y_stride=(channels + 4) * 4)
        return h.cpu().numpy(), y.cpu().numpy()

    h, y = run(ids, x)
    if tokens > 1:
        want, _ = orc.union_metadata(experts, selected, tokens, hidden, channels, ids.reshape(-1).tolist(), poison=0xFFFFFFFF)
        assert np.array_equal(w.union_meta.cpu().numpy().view(np.uint32), np.asarray(want, dtype=np.uint32))
    ref_h, ref_y = orc.moe_routed_reference(12, dn, gate, up, down, channels, hidden, experts, ids.reshape(-1), tokens, selected,
                                            np.ascontiguousarray(x[:, 1:]), stage=0, threads=8)
    assert nmse(h[:, :hidden], ref_h) <= 1e-12 and nmse(y[:, :channels], ref_y) <= 1e-12
    assert (h[:, hidden:] == -5.0).all() and (y[:, channels:] == -6.0).all() and gpu.error() == 0
    for pad in (1, 4) if dn == 14 else (1,):
        if pad != 1:
            h, y = run(ids, x, pad)
            _, ref_y = orc.moe_routed_reference(12, dn, gate, up, down, channels, hidden, experts, ids.reshape(-1), tokens, selected,
                                                np.ascontiguousarray(x[:, 1:]), stage=8, threads=8)
            assert nmse(h[:, :hidden], ref_h) <= 1e-12 and nmse(y[:, :channels], ref_y) <= 1e-12 and gpu.error() == 0
        if tokens > 2:
            part_h, part_y = run(ids[-2:], np.ascontiguousarray(x[-2:]), pad)
            assert np.array_equal(part_h, h[routes - 2 * selected:]) and np.array_equal(part_y, y[routes - 2 * selected:])


@pytest.mark.parametrize("tokens", [1, 2, 3])
def test_routed_m8_largest_rows(gpu, tsp, orc, synth, tokens):
    """Rows near the largest float, whose sums with the codes pass it before the block scales bring them back: finite results, no error. The
    gates are all minima, below -1e30, and close; only the always-on sum of the up product has to hold."""
    channels, hidden, experts = 2048, 64, 4
    gate, up = synth.matrix(12, 99, hidden * experts, channels), synth.matrix(12, 100, hidden * experts, channels)
    tiny = np.array([2.0 ** -24], dtype=np.float16).view(np.uint8)
    gate.reshape(-1, 144)[:, 0:2] = 0
    gate.reshape(-1, 144)[:, 2:4] = tiny
    up.reshape(-1, 144)[:, 0:2] = tiny
    up.reshape(-1, 144)[:, 2:4] = 0
    w = tsp.PlanarMoeWeights(gpu, 12, 8, channels, hidden, experts, gate, up, synth.matrix(8, 101, channels * experts, hidden))
    x = np.full((tokens, channels), 3e37, dtype=np.float32)
    x[-1] = 1.0  # an ordinary row beside them
    x[0, 7] = 1e37
    if tokens == 1:
        x[0] = 3e37
    h, y = tsp.planar_moe_routed_m8(gpu, w, gpu.upload(np.array([[1, 2]] * tokens, dtype=np.uint32).reshape(-1)), gpu.upload(x), tokens, 2)
    h, y = h.cpu().numpy(), y.cpu().numpy()
    assert gpu.error() == 0 and np.isfinite(h).all() and np.isfinite(y).all()
    if tokens > 1:
        ref_h, _ = orc.moe_routed_reference(12, 8, gate, up, synth.matrix(8, 101, channels * experts, hidden), channels, hidden, experts,
                                            np.array([1, 2], dtype=np.uint32), 1, 2, x[-1:], threads=4)
        assert nmse(h[-2:], ref_h) <= 1e-12
