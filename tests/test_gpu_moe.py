"""GPU parity of the MoE expert path (routing, grouped expert matmuls, activation, combination) against
the CPU oracle, through the C ABI. Shapes follow the reference's tests (src/moe.rs:1135-1219: 6 experts,
top-3; src/cuda.rs:2145-2179) with widths that are whole MLX groups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4_0, Q8_0, Q4_K, Q5_K, Q6_K, MXFP4 = 2, 8, 12, 13, 14, 39


@pytest.fixture(scope="module")
def be():
    from oxinfer_amd import HipBackend
    b = HipBackend(0)
    yield b
    b.close()


def row_err(y, ref):
    m = np.maximum(np.abs(ref).max(axis=1), 1e-30)
    return float((np.abs(y - ref).max(axis=1) / m).max())


def make_routes(oxref, t, ne, k, seed):
    from oxinfer_amd import synth
    logits = synth.router_logits(t, ne, seed)
    idx = np.zeros((t, k), np.uint32)
    w = np.zeros((t, k), np.float32)
    for i in range(t):
        idx[i], w[i] = oxref.route_top_k(logits[i], k)
    return logits, idx, w


def test_route_top_k_matches_oracle_and_definition(be, oxref):
    import torch
    from oxinfer_amd import synth
    t, ne, k = 33, 128, 8
    logits = synth.router_logits(t, ne, 5)
    logits[0, 7] = logits[0, 90] = logits[0].max() + 1.0   # a tie at the top: the lower index first
    logits[1, :] = 0.25                                      # all equal: indices 0..k-1
    logits[2, 3] = -0.0
    logits[2, 4] = 0.0                                       # total order: +0.0 above -0.0
    idx, w = be.route_top_k(torch.from_numpy(logits).cuda(), k)
    idx, w = idx.cpu().numpy().astype(np.uint32), w.cpu().numpy()
    for i in range(t):
        ri, rw = oxref.route_top_k(logits[i], k)
        assert np.array_equal(idx[i], ri), i
        assert np.allclose(w[i], rw, rtol=1e-6, atol=0)
        # the definition: softmax over all experts, the k largest, renormalized
        p = np.exp(logits[i].astype(np.float64) - logits[i].max())
        p /= p.sum()
        top = p[ri] / p[ri].sum()
        assert np.allclose(rw, top, rtol=1e-5)
    assert list(idx[0, :2]) == [7, 90] and list(idx[1]) == list(range(k))


@pytest.mark.parametrize("ne,k", [(100, 4), (256, 8), (300, 6), (64, 1), (33, 32), (7, 7), (1024, 16)])
def test_route_top_k_other_sizes(be, oxref, ne, k):
    """Up to 256 experts the kernel counts ranks, beyond that it runs k rounds of argmax: both against the oracle, with
    ties (quantized logits) and expert counts that do not fill the lanes."""
    import torch
    from oxinfer_amd import synth
    t = 9
    logits = synth.router_logits(t, ne, 40 + ne)
    logits[3:6] = np.round(logits[3:6] * 2.0) / 2.0  # many ties
    idx, w = be.route_top_k(torch.from_numpy(logits).cuda(), k)
    idx, w = idx.cpu().numpy().astype(np.uint32), w.cpu().numpy()
    for i in range(t):
        ri, rw = oxref.route_top_k(logits[i], k)
        assert np.array_equal(idx[i], ri), i
        assert np.allclose(w[i], rw, rtol=1e-6, atol=0), i


def moe_reference(oxref, kind, gate_up, down, h, inter, x, idx, w, y0, down_kind=None):
    """Each (token, route) pair on the oracle's decode kernels, combined in route order (what
    forward_batched computes row by row, src/moe.rs:438-617)."""
    y = y0.copy()
    t, k = idx.shape
    for i in range(t):
        for j in range(k):
            e = int(idx[i, j])
            if kind == "mlx":
                gu = oxref.q4_decode(*gate_up[e], 64, 2 * inter, h, x[i], 1)[0]
            else:
                gu = oxref.gguf_decode(kind, gate_up[e], 2 * inter, h, x[i], 1)[0]
            a = oxref.silu_mul(gu[:inter], gu[inter:])
            if kind == "mlx":
                o = oxref.q4_decode(*down[e], 64, h, inter, a, 1)[0]
            else:
                o = oxref.gguf_decode(down_kind or kind, down[e], h, inter, a, 1)[0]
            y[i] = y[i] + w[i, j] * o
    return y


@pytest.fixture(scope="module")
def mlx_experts(oxref):
    from oxinfer_amd import synth
    ne, h, inter = 6, 256, 128
    raw_gu = [synth.mlx_q4(2 * inter, h, 100 + e) for e in range(ne)]
    raw_dn = [synth.mlx_q4(h, inter, 200 + e) for e in range(ne)]
    q_gu = [oxref.from_mlx_q4(*r, 2 * inter, h, 64) for r in raw_gu]
    q_dn = [oxref.from_mlx_q4(*r, h, inter, 64) for r in raw_dn]
    return ne, h, inter, raw_gu, raw_dn, q_gu, q_dn


def test_moe_mlx_matches_oracle(be, oxref, mlx_experts):
    from oxinfer_amd import synth
    ne, h, inter, raw_gu, raw_dn, q_gu, q_dn = mlx_experts
    k = 3
    dev = be.upload_moe([be.desc_mlx_q4(*r, 64, 2 * inter, h) for r in raw_gu], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_dn], h, inter)
    assert dev is not None, be.last_error()
    from oxinfer_amd import hip
    for t in (1, 2, 5, 7, 8, 19, 40):
        x = synth.activations(t, h, 300 + t)
        _, idx, w = make_routes(oxref, t, ne, k, 400 + t)
        y0 = synth.activations(t, h, 500 + t)  # the call adds into y
        ref = moe_reference(oxref, "mlx", q_gu, q_dn, h, inter, x, idx, w, y0)
        # the oracle's own MoE driver agrees with the composition above (decode path)
        ref2 = oxref.moe_q4(q_gu, q_dn, 64, h, inter, x, t, idx, w, y0, decode_path=True)
        assert np.array_equal(ref2.view(np.uint32), ref.view(np.uint32))
        # from 8 tokens on the CPU takes its grouped f32 path (exact activations, Act::scalar)
        ref3 = oxref.moe_q4(q_gu, q_dn, 64, h, inter, x, t, idx, w, y0, decode_path=False) if t >= 8 else None
        # the integer path (int8 activations, the decode kernels' semantics) at every size
        dev.set_mode(hip.MOE_INT8)
        try:
            y = y0.copy()
            assert be.moe(x, t, h, inter, idx, w, k, dev, y), be.last_error()
        finally:
            dev.set_mode(hip.MOE_AUTO)
        assert row_err(y - y0, ref - y0) < 1e-3, t
        if ref3 is not None:
            # int8 activations against the exact product: within the reference's own bound for them (3e-2, src/ggml.rs:1904)
            assert row_err(y - y0, ref3 - y0) < 3e-2, t
        # the library's own choice: with six or more routed rows per expert the bf16 form of the grouped matmuls, which
        # is the grouped f32 path up to the bf16 rounding of x and of the activation's output (2^-9 per element, which
        # these short rows of 256 and 128 barely average; the bar for the bf16 matrix cores is 2e-2)
        y = y0.copy()
        assert be.moe(x, t, h, inter, idx, w, k, dev, y), be.last_error()
        if (t * k) // ne >= 6:
            assert row_err(y - y0, ref3 - y0) < 1e-2, t
            # with activations that are bf16 values already (the prefill workload's) only the intermediate is rounded
            import torch
            xb = torch.from_numpy(x).to(torch.bfloat16).to(torch.float32).numpy()
            refb = oxref.moe_q4(q_gu, q_dn, 64, h, inter, xb, t, idx, w, y0, decode_path=False)
            yb = y0.copy()
            assert be.moe(xb, t, h, inter, idx, w, k, dev, yb), be.last_error()
            assert row_err(yb - y0, refb - y0) < 4e-3, t
        else:
            assert row_err(y - y0, ref - y0) < 1e-3, t


def test_moe_batched_equals_one_at_a_time(be, oxref, mlx_experts):
    """src/moe.rs:1135-1219: every token's row is bit-identical whether it runs alone or in a batch."""
    from oxinfer_amd import synth
    ne, h, inter, raw_gu, raw_dn, _, _ = mlx_experts
    k, t = 3, 7
    dev = be.upload_moe([be.desc_mlx_q4(*r, 64, 2 * inter, h) for r in raw_gu], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_dn], h, inter)
    x = synth.activations(t, h, 1)
    _, idx, w = make_routes(oxref, t, ne, k, 2)
    y = np.zeros((t, h), np.float32)
    assert be.moe(x, t, h, inter, idx, w, k, dev, y)
    for i in range(t):
        y1 = np.zeros((1, h), np.float32)
        assert be.moe(x[i:i + 1], 1, h, inter, idx[i:i + 1], w[i:i + 1], k, dev, y1)
        assert np.array_equal(y1[0].view(np.uint32), y[i].view(np.uint32)), i


def moe_grouped_reference(oxref, kind, gate_up, down, h, inter, x, idx, w, y0):
    """The grouped prefill path over GGUF experts (src/moe.rs:735-827): per (token, route) the f32 product of the
    dequantized rows (matmul_quant_grouped, src/kernels.rs:195-279), Act::scalar (libm exp) between the two, combined in
    route order."""
    y = y0.copy()
    t, k = idx.shape
    for i in range(t):
        for j in range(k):
            e = int(idx[i, j])
            gu = oxref.gemm_quant(kind, gate_up[e], None, None, 2 * inter, h, x[i:i + 1], 1, threads=1)[0]
            g, u = gu[:inter], gu[inter:]
            with np.errstate(over="ignore"):  # exp overflows to inf for very negative gates: the quotient is -0.0, as on the device
                a = (g / (np.float32(1.0) + np.exp(-g, dtype=np.float32)) * u).astype(np.float32)
            o = oxref.gemm_quant(kind, down[e], None, None, h, inter, a[None, :], 1, threads=1)[0]
            y[i] = y[i] + w[i, j] * o
    return y


@pytest.mark.parametrize("kind", [Q4_0, Q8_0, Q4_K, MXFP4])
def test_moe_gguf_experts(be, oxref, kind):
    """GGUF experts: decode-sized passes on the integer kernels against the decode semantics (1e-3). At prefill size (40
    tokens, twenty routed rows per expert) they take the reference's grouped form on the bf16 matrix cores: within 2e-2 of
    the grouped f32 path (src/moe.rs:735-827; 6e-3 when the activations are bf16 values already), and the integer kernels
    (OXHIP_MOE_INT8) within 1e-3 of the decode semantics."""
    from oxinfer_amd import hip, synth
    ne, h, inter, k = 4, 256, 256, 2
    gu = [oxref.random_blocks(kind, 2 * inter * h // oxref.block_size(kind), 10 + e)[0] for e in range(ne)]
    dn = [oxref.random_blocks(kind, h * inter // oxref.block_size(kind), 20 + e)[0] for e in range(ne)]
    dev = be.upload_moe([be.desc_gguf(kind, g, 2 * inter, h) for g in gu], [be.desc_gguf(kind, d, h, inter) for d in dn], h, inter)
    assert dev is not None, be.last_error()
    for t in (1, 3, 11, 40):  # (40: twenty rows per expert)
        x = synth.activations(t, h, 30 + t)
        _, idx, w = make_routes(oxref, t, ne, k, 40 + t)
        zero = np.zeros((t, h), np.float32)
        ref = moe_reference(oxref, kind, gu, dn, h, inter, x, idx, w, zero)
        y = np.zeros((t, h), np.float32)
        assert be.moe(x, t, h, inter, idx, w, k, dev, y), be.last_error()
        if t == 40:
            grouped = moe_grouped_reference(oxref, kind, gu, dn, h, inter, x, idx, w, zero)
            assert row_err(y, grouped) < 2e-2, (t, row_err(y, grouped))
            assert row_err(y, ref) > 1e-5   # (not the integer kernels' rows: the bf16 form did run)
            xb = synth.bf16_round(x)         # activations that are bf16 values already: only the intermediate is rounded
            yb = np.zeros((t, h), np.float32)
            assert be.moe(xb, t, h, inter, idx, w, k, dev, yb), be.last_error()
            assert row_err(yb, moe_grouped_reference(oxref, kind, gu, dn, h, inter, xb, idx, w, zero)) < 6e-3
            dev.set_mode(hip.MOE_INT8)
            try:
                y = np.zeros((t, h), np.float32)
                assert be.moe(x, t, h, inter, idx, w, k, dev, y), be.last_error()
            finally:
                dev.set_mode(hip.MOE_AUTO)
        assert row_err(y, ref) < 1e-3, t


def test_moe_prefill_rows_do_not_depend_on_the_batch(be, oxref, mlx_experts):
    """In the bf16 form too every (token, row) sum is formed on its own in a fixed order: a token's output is
    bit-identical whichever other tokens share the pass (and its expert's chunks). (Where the launches split K over the same number of
    waves, here none: that number goes by the pass's size, and the order of a sum's terms with it.)"""
    from oxinfer_amd import synth
    ne, h, inter, raw_gu, raw_dn, _, _ = mlx_experts
    k, t = 3, 40
    dev = be.upload_moe([be.desc_mlx_q4(*r, 64, 2 * inter, h) for r in raw_gu], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_dn], h, inter)
    x = synth.activations(t, h, 21)
    _, idx, w = make_routes(oxref, t, ne, k, 22)
    y = np.zeros((t, h), np.float32)
    assert be.moe(x, t, h, inter, idx, w, k, dev, y)
    for keep in (np.arange(8, 40), np.arange(0, 40, 2)[:14].repeat(1), np.r_[0:5, 20:33]):
        assert (len(keep) * k) // ne >= 6  # still the bf16 form
        ys = np.zeros((len(keep), h), np.float32)
        assert be.moe(np.ascontiguousarray(x[keep]), len(keep), h, inter, np.ascontiguousarray(idx[keep]), np.ascontiguousarray(w[keep]), k, dev, ys)
        assert np.array_equal(ys.view(np.uint32), y[keep].view(np.uint32))


# staged in three phases and one, an odd number of steps; one; four and one; three row tiles per wave in the down launch; two, three (the last
# ending past the matrix) and four runs of row tiles per workgroup there, three row tiles per wave in the gate / up launch, the last group
# ragged (24 copies) or not (32). tests/test_moe_plan.py holds them to that.
CHUNK_SIZES = [(2304, 384, 1), (256, 256, 1), (4096, 256, 1), (2048, 384, 14), (2048, 384, 16), (2048, 512, 24), (2048, 384, 32)]
CHUNK_ROWS = [33, 32, 17, 16, 1]  # of the experts


@pytest.mark.parametrize("fmt", ["mlx", "Q4_K", "Q8_0", "Q4_0", "MXFP4", "mlx, Q8_0 down"])
@pytest.mark.parametrize("h,inter,copies", CHUNK_SIZES)
def test_moe_prefill_chunks(be, oxref, fmt, h, inter, copies):
    """The bf16 form's chunks at the edges of its token tiles and of a chunk (experts of 33, 32, 17, 16 and 1 rows): within 6e-3 of the
    reference's grouped f32 path on activations that are bf16 values already (as in test_moe_gguf_experts), and bit for bit the same
    where the tokens, and with them the rows' places, come in another order."""
    from oxinfer_amd import synth
    if fmt == "Q4_K":
        inter = (inter + 255) // 256 * 256  # whole super-blocks
    rows = CHUNK_ROWS
    ne, t = len(rows), sum(rows)
    kinds = {"Q4_K": (Q4_K, synth.gguf_q4_k), "Q8_0": (Q8_0, synth.gguf_q8_0), "Q4_0": (Q4_0, synth.gguf_q4_0), "MXFP4": (MXFP4, synth.gguf_mxfp4)}

    def experts(f, n, c, seed):
        """(raw, dequantized f32 rows, descriptor) of each expert"""
        out = []
        for e in range(ne):
            if f == "mlx":
                raw = synth.mlx_q4(n, c, seed + e)
                out.append((raw, oxref.dequant_rows_q4(*oxref.from_mlx_q4(*raw, n, c, 64), 64, n, c), be.desc_mlx_q4(*raw, 64, n, c)))
            else:
                kind, make = kinds[f]
                raw = make(n, c, seed + e)
                out.append((raw, oxref.dequantize_rows(kind, raw, n, c), be.desc_gguf(kind, raw, n, c)))
        return out

    first, second = ("mlx", "Q8_0") if "down" in fmt else (fmt, fmt)
    gu, dn = experts(first, 2 * inter, h, 2500), experts(second, h, inter, 2600)
    dev = be.upload_moe([e[2] for e in gu] * copies, [e[2] for e in dn] * copies, h, inter)
    assert dev is not None, be.last_error()
    t *= copies
    idx = np.repeat(np.arange(ne * copies, dtype=np.uint32), rows * copies)[:, None]
    w = np.ones((t, 1), np.float32)
    x = synth.bf16_round(synth.activations(t, h, 2700))
    ref = np.zeros((t, h))
    for e in range(ne):
        at = idx[:, 0] % ne == e
        p = x[at].astype(np.float64) @ gu[e][1].astype(np.float64).T
        g, u = p[:, :inter], p[:, inter:]
        ref[at] = (g / (1.0 + np.exp(-g)) * u) @ dn[e][1].astype(np.float64).T
    results = []
    for order in (np.arange(t), np.random.default_rng(5).permutation(t)):
        y = np.zeros((t, h), np.float32)
        assert be.moe(np.ascontiguousarray(x[order]), t, h, inter, np.ascontiguousarray(idx[order]), w, 1, dev, y), be.last_error()
        back = np.zeros_like(y)
        back[order] = y
        results.append(back)
    assert row_err(results[0], ref.astype(np.float32)) < 6e-3
    assert np.array_equal(results[0].view(np.uint32), results[1].view(np.uint32))


@pytest.mark.parametrize("fmt", ["mlx", "Q4_K", "Q8_0", "Q4_0", "MXFP4"])
def test_moe_few_rows_per_expert(be, oxref, fmt):
    """A launch's chunks of up to four rows run in another form than its longer ones, and below three routed rows per expert the
    activation is in the gate / up launch: on both sides of these lines, one expert having every token (chunks of eight, a ragged
    last one), each token's row is bit for bit what it is alone."""
    from oxinfer_amd import synth
    ne, h, inter, k = 16, 512, 256, 2
    if fmt == "mlx":
        descs = [[be.desc_mlx_q4(*synth.mlx_q4(n, c, s + e), 64, n, c) for e in range(ne)] for n, c, s in ((2 * inter, h, 2100), (h, inter, 2200))]
    else:
        kind, make = {"Q4_K": (Q4_K, synth.gguf_q4_k), "Q8_0": (Q8_0, synth.gguf_q8_0), "Q4_0": (Q4_0, synth.gguf_q4_0), "MXFP4": (MXFP4, synth.gguf_mxfp4)}[fmt]
        descs = [[be.desc_gguf(kind, make(n, c, s + e), n, c) for e in range(ne)] for n, c, s in ((2 * inter, h, 2100), (h, inter, 2200))]
    dev = be.upload_moe(*descs, h, inter)
    assert dev is not None, be.last_error()
    for t in (5, 8, 9, 23, 24):  # 46 routed rows over 16 experts: the last pass under the line
        x = synth.activations(t, h, 2300 + t)
        _, idx, w = make_routes(oxref, t, ne, k, 2400 + t)
        other = np.where(idx[:, 1] == 0, 1, idx[:, 1])
        idx = np.ascontiguousarray(np.stack([np.zeros_like(other), other], 1))
        y = np.zeros((t, h), np.float32)
        assert be.moe(x, t, h, inter, idx, w, k, dev, y), be.last_error()
        for i in range(t):
            y1 = np.zeros((1, h), np.float32)
            assert be.moe(x[i:i + 1], 1, h, inter, idx[i:i + 1], w[i:i + 1], k, dev, y1)
            assert np.array_equal(y1[0].view(np.uint32), y[i].view(np.uint32)), (t, i)


def test_moe_rows_too_long_for_eight_at_once(be, oxref):
    """Rows of 90112 columns: the staged scales of eight routed rows are more than LDS holds, those of four are not."""
    from oxinfer_amd import synth
    ne, h, inter = 2, 90112, 32
    layer = be.upload_moe([be.desc_mlx_q4(*synth.mlx_q4(2 * inter, h, 2900 + e), 64, 2 * inter, h) for e in range(ne)],
                          [be.desc_gguf(Q8_0, synth.gguf_q8_0(h, inter, 2910 + e), h, inter) for e in range(ne)], h, inter)
    assert layer is not None, be.last_error()
    x, idx, w = synth.activations(5, h, 2920), np.array([[0], [0], [0], [1], [0]], np.uint32), np.ones((5, 1), np.float32)
    y = np.zeros((5, h), np.float32)
    assert be.moe(x, 5, h, inter, idx, w, 1, layer, y), be.last_error()
    for i in range(5):
        y1 = np.zeros((1, h), np.float32)
        assert be.moe(x[i:i + 1], 1, h, inter, idx[i:i + 1], w[i:i + 1], 1, layer, y1), be.last_error()
        assert np.array_equal(y1[0].view(np.uint32), y[i].view(np.uint32)), i


@pytest.mark.parametrize("t", [1, 3, 11, 40])  # one token's three launches; the activation in the gate / up launch; above six tokens per expert not
@pytest.mark.parametrize("split", [False, True])
def test_moe_activation_of_nans_has_no_scale(be, oxref, t, split):
    """Q4_K gate and up rows of a token with a NaN are NaN throughout; the activation's blocks then have the scale 0 (as the oracle
    has it), which Q8_0 down matrices turn into zeros. The other tokens' rows are what they are without it."""
    from oxinfer_amd import synth
    ne, h, inter, k = 12, 256, 128, 2
    gu = [synth.gguf_q4_k(2 * inter, h, 2500 + e) for e in range(ne)]
    dn = [synth.gguf_q8_0(h, inter, 2600 + e) for e in range(ne)]
    down = [be.desc_gguf(Q8_0, d, h, inter) for d in dn]
    if split:
        halves = [(np.ascontiguousarray(g.reshape(2, -1)[0]), np.ascontiguousarray(g.reshape(2, -1)[1])) for g in gu]
        layer = be.upload_moe([be.desc_gguf(Q4_K, g, inter, h) for g, _ in halves], down, h, inter, up=[be.desc_gguf(Q4_K, u, inter, h) for _, u in halves])
    else:
        layer = be.upload_moe([be.desc_gguf(Q4_K, g, 2 * inter, h) for g in gu], down, h, inter)
    assert layer is not None, be.last_error()
    x = synth.activations(t, h, 2700 + t)
    _, idx, w = make_routes(oxref, t, ne, k, 2800 + t)
    from oxinfer_amd import hip
    layer.set_mode(hip.MOE_INT8)
    y, clean = np.zeros((t, h), np.float32), np.zeros((t, h), np.float32)
    assert be.moe(x, t, h, inter, idx, w, k, layer, clean), be.last_error()
    x[t // 2, 5] = np.nan
    assert np.array_equal(moe_reference(oxref, Q4_K, gu, dn, h, inter, x[t // 2:t // 2 + 1], idx[t // 2:t // 2 + 1], w[t // 2:t // 2 + 1], np.zeros((1, h), np.float32), Q8_0),
                          np.zeros((1, h)))
    assert be.moe(x, t, h, inter, idx, w, k, layer, y), be.last_error()
    assert not y[t // 2].any()
    keep = np.arange(t) != t // 2
    assert np.array_equal(y[keep].view(np.uint32), clean[keep].view(np.uint32))


def test_moe_config_shapes(be, oxref):
    """The benchmark's expert shapes (h 2048, inter 768, top-8) over 16 experts: one token on the integer kernels against
    the oracle's decode path, 32 tokens (16 routed rows per expert: the bf16 form) against its grouped f32 path."""
    import torch
    from oxinfer_amd import synth
    ne, h, inter, k = 16, 2048, 768, 8
    raw_gu = [synth.mlx_q4(2 * inter, h, 700 + e) for e in range(ne)]
    raw_dn = [synth.mlx_q4(h, inter, 800 + e) for e in range(ne)]
    q_gu = [oxref.from_mlx_q4(*r, 2 * inter, h, 64) for r in raw_gu]
    q_dn = [oxref.from_mlx_q4(*r, h, inter, 64) for r in raw_dn]
    dev = be.upload_moe([be.desc_mlx_q4(*r, 64, 2 * inter, h) for r in raw_gu], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_dn], h, inter)
    assert dev is not None, be.last_error()
    for t, decode_path, tol in ((1, True, 1e-3), (32, False, 5e-3)):
        x = synth.activations(t, h, 900 + t, bf16=True)  # bf16 values, as in the workload
        _, idx, w = make_routes(oxref, t, ne, k, 950 + t)
        y0 = np.zeros((t, h), np.float32)
        y = y0.copy()
        assert be.moe(x, t, h, inter, idx, w, k, dev, y), be.last_error()
        ref = oxref.moe_q4(q_gu, q_dn, 64, h, inter, x, t, idx, w, y0, decode_path=decode_path)
        assert row_err(y, ref) < tol, (t, row_err(y, ref))


@pytest.fixture(scope="module")
def config_experts(oxref):
    """128 experts of [1536, 2048] + [2048, 768], MLX 4-bit g64."""
    from oxinfer_amd import synth
    ne, h, inter = 128, 2048, 768
    raw_gu = [synth.mlx_q4(2 * inter, h, 1100 + e) for e in range(ne)]
    raw_dn = [synth.mlx_q4(h, inter, 1300 + e) for e in range(ne)]
    q_gu = [oxref.from_mlx_q4(*r, 2 * inter, h, 64) for r in raw_gu]
    q_dn = [oxref.from_mlx_q4(*r, h, inter, 64) for r in raw_dn]
    return ne, h, inter, raw_gu, raw_dn, q_gu, q_dn


def test_moe_config_128_experts(be, oxref, config_experts):
    """BASELINE configs[3] at its full size: 128 experts, top-8, h 2048, inter 768, bf16-valued activations, routing
    on the device. T = 1 (8 experts, the integer kernels) against the oracle's decode path (forward_batched,
    src/moe.rs:438-617) within 1e-3; T = 256 (2048 routed rows, 16 per expert on average: the bf16 form) against the
    grouped f32 path (src/moe.rs:735-827) on a sample of tokens (a token's row depends on its own routes only) within
    1e-2, and the integer kernels at that size within the reference's bound for int8 activations (3e-2, src/ggml.rs:1904)."""
    import torch
    from oxinfer_amd import hip, synth
    ne, h, inter, raw_gu, raw_dn, q_gu, q_dn = config_experts
    k = 8
    dev = be.upload_moe([be.desc_mlx_q4(*r, 64, 2 * inter, h) for r in raw_gu], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_dn], h, inter)
    assert dev is not None, be.last_error()
    for t in (1, 256):
        x = synth.activations(t, h, 1500 + t, bf16=True)
        logits = synth.router_logits(t, ne, 1600 + t)
        idx_d, w_d = be.route_top_k(torch.from_numpy(logits).cuda(), k)
        idx, w = idx_d.cpu().numpy().astype(np.uint32), w_d.cpu().numpy()
        for i in range(t):  # the device's routing is the oracle's (src/moe.rs:180-193)
            ri, rw = oxref.route_top_k(logits[i], k)
            assert np.array_equal(idx[i], ri) and np.allclose(w[i], rw, rtol=1e-6, atol=0)
        y = torch.zeros((t, h), dtype=torch.float32, device="cuda")
        be.dev_moe(dev, torch.from_numpy(x).cuda(), idx_d, w_d, y)
        y = y.cpu().numpy()
        # routing inside the pass (one call: top-k of the logits, then the experts): the same routes and the same rows
        y2 = torch.zeros((t, h), dtype=torch.float32, device="cuda")
        sel = be.moe_routed(dev, torch.from_numpy(x).cuda(), torch.from_numpy(logits).cuda(), k, y2).cpu().numpy()
        assert np.array_equal(sel[0].view(np.uint32), idx) and np.array_equal(sel[1].view(np.float32).view(np.uint32), w.view(np.uint32))
        assert np.array_equal(y2.cpu().numpy().view(np.uint32), y.view(np.uint32))
        sample = np.arange(t) if t == 1 else np.r_[0:3, 100:103, 253:256, np.random.default_rng(5).integers(0, t, 7)]
        xs, si, sw = np.ascontiguousarray(x[sample]), np.ascontiguousarray(idx[sample]), np.ascontiguousarray(w[sample])
        y0 = np.zeros((len(sample), h), np.float32)
        if t == 1:
            ref = oxref.moe_q4(q_gu, q_dn, 64, h, inter, xs, 1, si, sw, y0, decode_path=True)
            assert row_err(y, ref) < 1e-3, row_err(y, ref)
        else:
            assert len(set(idx.reshape(-1).tolist())) == ne  # every expert is in use
            ref = oxref.moe_q4(q_gu, q_dn, 64, h, inter, xs, len(sample), si, sw, y0, decode_path=False)
            assert row_err(y[sample], ref) < 1e-2, row_err(y[sample], ref)
            dev.set_mode(hip.MOE_INT8)
            try:
                yi = torch.zeros((t, h), dtype=torch.float32, device="cuda")
                be.dev_moe(dev, torch.from_numpy(x).cuda(), idx_d, w_d, yi)
                yi = yi.cpu().numpy()
            finally:
                dev.set_mode(hip.MOE_AUTO)
            assert row_err(yi[sample], ref) < 3e-2
            refi = oxref.moe_q4(q_gu, q_dn, 64, h, inter, xs[:4], 4, si[:4], sw[:4], y0[:4], decode_path=True)
            assert row_err(yi[sample[:4]], refi) < 1e-3


def test_moe_long_rows_take_smaller_chunks(be, oxref):
    """Experts of the Llama-8B MLP shape (h 4096, inter 14336) in GGUF Q8_0: a prefill-sized pass (20 routed rows per
    expert and more) would take chunks of 32 rows, whose staged activations do not fit the LDS at these row lengths;
    the pass must still run on the device, on smaller chunks, and match the oracle's decode kernels row by row."""
    from oxinfer_amd import synth
    ne, h, inter, k, t = 2, 4096, 14336, 2, 24
    gu = [synth.gguf_q8_0(2 * inter, h, 2100 + e) for e in range(ne)]
    dn = [synth.gguf_q8_0(h, inter, 2200 + e) for e in range(ne)]
    dev = be.upload_moe([be.desc_gguf(Q8_0, g, 2 * inter, h) for g in gu], [be.desc_gguf(Q8_0, d, h, inter) for d in dn], h, inter)
    assert dev is not None, be.last_error()
    x = synth.activations(t, h, 2300)
    idx = np.tile(np.array([[0, 1]], np.uint32), (t, 1))
    w = np.tile(np.array([[0.75, 0.25]], np.float32), (t, 1))
    y = np.zeros((t, h), np.float32)
    assert be.moe(x, t, h, inter, idx, w, k, dev, y), be.last_error()
    sample = [0, 7, 23]
    ref = moe_reference(oxref, Q8_0, gu, dn, h, inter, x[sample], idx[sample], w[sample], np.zeros((len(sample), h), np.float32))
    assert row_err(y[sample], ref) < 1e-3


def test_moe_duplicate_routes_within_a_token(be, oxref, mlx_experts):
    """Routes that name one expert several times (nothing in Backend::moe forbids them): one token whose eight routes all
    go to expert 0 cuts eight one-row chunks, more than there are experts."""
    from oxinfer_amd import synth
    ne, h, inter, raw_gu, raw_dn, q_gu, q_dn = mlx_experts
    dev = be.upload_moe([be.desc_mlx_q4(*r, 64, 2 * inter, h) for r in raw_gu], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_dn], h, inter)
    x = synth.activations(1, h, 77)
    idx = np.zeros((1, 8), np.uint32)
    w = np.full((1, 8), 0.125, np.float32)
    y = np.zeros((1, h), np.float32)
    assert be.moe(x, 1, h, inter, idx, w, 8, dev, y), be.last_error()
    ref = moe_reference(oxref, "mlx", q_gu, q_dn, h, inter, x, idx, w, np.zeros((1, h), np.float32))
    assert row_err(y, ref) < 1e-3


@pytest.mark.parametrize("act,param", [(1, 0.0), (2, 0.1)])   # MoeAct::GeluTanh, MoeAct::SiluClamp(0.1)
@pytest.mark.parametrize("split", [False, True])               # fused [2 inter, h] experts / separate gate and up
def test_moe_activation_kinds_and_split_experts(be, oxref, act, param, split):
    """MoeAct::GeluTanh and SiluClamp(l), and experts uploaded as separate gate / up matrices (src/gpu.rs:35-54,
    :206-216), at decode sizes (the integer kernels against Experts::forward_batched's semantics, 1e-3) and at a prefill
    size (40 tokens: fused experts take the bf16 form against the grouped f32 path with Act::scalar, 1e-2; split experts
    stay on the integer kernels: 1e-3 of the decode semantics, 5e-2 of the exact product on these short rows). The clamp limit lies inside
    the products' range, so a missing clamp fails."""
    from oxinfer_amd import synth
    ne, h, inter, k = 6, 256, 128, 3
    raw_g = [synth.mlx_q4(inter, h, 3100 + e) for e in range(ne)]
    raw_u = [synth.mlx_q4(inter, h, 3200 + e) for e in range(ne)]
    raw_d = [synth.mlx_q4(h, inter, 3300 + e) for e in range(ne)]
    raw_gu = [tuple(np.concatenate([a, b]) for a, b in zip(raw_g[e], raw_u[e])) for e in range(ne)]
    q_gu = [oxref.from_mlx_q4(*r, 2 * inter, h, 64) for r in raw_gu]
    q_d = [oxref.from_mlx_q4(*r, h, inter, 64) for r in raw_d]
    if split:
        dev = be.upload_moe([be.desc_mlx_q4(*r, 64, inter, h) for r in raw_g], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_d], h, inter,
                            up=[be.desc_mlx_q4(*r, 64, inter, h) for r in raw_u], act=act, act_param=param)
    else:
        dev = be.upload_moe([be.desc_mlx_q4(*r, 64, 2 * inter, h) for r in raw_gu], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_d], h, inter,
                            act=act, act_param=param)
    assert dev is not None, be.last_error()
    for t in (1, 3, 8, 40):
        x = synth.activations(t, h, 3400 + t)
        _, idx, w = make_routes(oxref, t, ne, k, 3500 + t)
        y0 = synth.activations(t, h, 3600 + t)
        y = y0.copy()
        assert be.moe(x, t, h, inter, idx, w, k, dev, y), be.last_error()
        dec = oxref.moe_q4(q_gu, q_d, 64, h, inter, x, t, idx, w, y0, decode_path=True, act=act, act_param=param)
        plain = oxref.moe_q4(q_gu, q_d, 64, h, inter, x, t, idx, w, y0, decode_path=True)
        assert row_err(plain - y0, dec - y0) > 2e-2          # the activation kind matters on these inputs
        if (t * k) // ne >= 6 and not split:
            grouped = oxref.moe_q4(q_gu, q_d, 64, h, inter, x, t, idx, w, y0, decode_path=False, act=act, act_param=param)
            assert row_err(y - y0, grouped - y0) < 1e-2, (t, row_err(y - y0, grouped - y0))
        else:
            assert row_err(y - y0, dec - y0) < 1e-3, (t, row_err(y - y0, dec - y0))
            if t >= 8:
                grouped = oxref.moe_q4(q_gu, q_d, 64, h, inter, x, t, idx, w, y0, decode_path=False, act=act, act_param=param)
                # int8 activations against the exact product: the reference's bound for them is 3e-2 on its own shapes
                # (src/ggml.rs:1904); these rows of 256 and 128 values average a little less
                assert row_err(y - y0, grouped - y0) < 5e-2, t


@pytest.mark.parametrize("act,param,split", [(1, 0.0, False), (2, 0.2, True)])
def test_moe_activation_kinds_config_shapes(be, oxref, act, param, split):
    """The same at the benchmark's expert shapes (h 2048, inter 768, top-8) over 16 experts: one token (decode) and 32
    tokens (16 routed rows per expert: the prefill size)."""
    from oxinfer_amd import synth
    ne, h, inter, k = 16, 2048, 768, 8
    raw_g = [synth.mlx_q4(inter, h, 4100 + e) for e in range(ne)]
    raw_u = [synth.mlx_q4(inter, h, 4200 + e) for e in range(ne)]
    raw_d = [synth.mlx_q4(h, inter, 4300 + e) for e in range(ne)]
    raw_gu = [tuple(np.concatenate([a, b]) for a, b in zip(raw_g[e], raw_u[e])) for e in range(ne)]
    q_gu = [oxref.from_mlx_q4(*r, 2 * inter, h, 64) for r in raw_gu]
    q_d = [oxref.from_mlx_q4(*r, h, inter, 64) for r in raw_d]
    if split:
        dev = be.upload_moe([be.desc_mlx_q4(*r, 64, inter, h) for r in raw_g], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_d], h, inter,
                            up=[be.desc_mlx_q4(*r, 64, inter, h) for r in raw_u], act=act, act_param=param)
    else:
        dev = be.upload_moe([be.desc_mlx_q4(*r, 64, 2 * inter, h) for r in raw_gu], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_d], h, inter,
                            act=act, act_param=param)
    assert dev is not None, be.last_error()
    for t in (1, 32):
        x = synth.activations(t, h, 4400 + t, bf16=True)
        _, idx, w = make_routes(oxref, t, ne, k, 4500 + t)
        y0 = np.zeros((t, h), np.float32)
        y = y0.copy()
        assert be.moe(x, t, h, inter, idx, w, k, dev, y), be.last_error()
        prefill_form = t == 32 and not split
        ref = oxref.moe_q4(q_gu, q_d, 64, h, inter, x, t, idx, w, y0, decode_path=not prefill_form, act=act, act_param=param)
        assert row_err(y, ref) < (5e-3 if prefill_form else 1e-3), (t, row_err(y, ref))


def test_moe_declines(be, oxref, mlx_experts):
    ne, h, inter, raw_gu, raw_dn, _, _ = mlx_experts
    dev = be.upload_moe([be.desc_mlx_q4(*r, 64, 2 * inter, h) for r in raw_gu], [be.desc_mlx_q4(*r, 64, h, inter) for r in raw_dn], h, inter)
    y = np.full((1, h), np.nan, np.float32)
    bad = np.array([[0, 1, ne]], np.uint32)  # a route past the experts (src/cuda.rs:803-813)
    assert not be.moe(np.zeros((1, h), np.float32), 1, h, inter, bad, np.ones((1, 3), np.float32), 3, dev, y)
    assert np.isnan(y).all() and "route" in be.last_error()
    # a CPU-only activation kind is declined at upload
    assert be.upload_moe([be.desc_mlx_q4(*raw_gu[0], 64, 2 * inter, h)], [be.desc_mlx_q4(*raw_dn[0], 64, h, inter)], h, inter, act=3) is None


def test_matvec_rows(be, oxref):
    """Backend::matvec_rows (src/gpu.rs:165): plain and silu(W x) * (U x) products, t in 1..=4."""
    n_out, n_in = 96, 512
    wk, _ = oxref.random_blocks(Q4_K, n_out * n_in // 256, 3)
    uk, _ = oxref.random_blocks(Q4_K, n_out * n_in // 256, 4)
    w, u = be.upload_gguf(Q4_K, wk, n_out, n_in), be.upload_gguf(Q4_K, uk, n_out, n_in)
    from oxinfer_amd import synth
    for t in (1, 4):
        x = synth.activations(t, n_in, 50 + t)
        y0, y1 = np.zeros((t, n_out), np.float32), np.zeros((t, n_out), np.float32)
        assert be.matvec_rows(x, t, n_in, [(w, None, y0), (w, u, y1)]), be.last_error()
        g = oxref.gguf_decode(Q4_K, wk, n_out, n_in, x, t)
        assert row_err(y0, g) < 1e-3
        ref = oxref.silu_mul(g, oxref.gguf_decode(Q4_K, uk, n_out, n_in, x, t))
        assert row_err(y1, ref) < 1e-3
    assert not be.matvec_rows(np.zeros((5, n_in), np.float32), 5, n_in, [(w, None, np.zeros((5, n_out), np.float32))])


@pytest.mark.parametrize("kind,n_out,n_in", [(Q4_K, 1000, 768), (Q8_0, 272, 14336), (Q4_K, 48, 14336),
                                             (Q6_K, 48, 3072), (Q8_0, 48, 5120), (Q4_0, 40, 5376), (Q4_K, 48, 5376), (Q5_K, 40, 5376)])
def test_matvec_rows_shares_a_launch_and_pairs_keep_the_bits(be, oxref, kind, n_out, n_in):
    """Several RowsJobs of one call (plain and gate / up) share one launch; a gate / up job's rows are silu_mul of the two
    products as separate plain jobs give them, bit for bit (K-sliced shapes and ragged row groups included; the last five have rows of
    eight runs, whose pairs' workgroups are sixteen waves)."""
    from oxinfer_amd import synth
    raws = [oxref.random_blocks(kind, n_out * n_in // oxref.block_size(kind), 70 + i)[0] for i in range(3)]
    ws = [be.upload_gguf(kind, r, n_out, n_in) for r in raws]
    for t in (1, 3, 4):
        x = synth.activations(t, n_in, 80 + t)
        ys = [np.zeros((t, n_out), np.float32) for _ in range(5)]
        assert be.matvec_rows(x, t, n_in, [(ws[0], None, ys[0]), (ws[0], ws[1], ys[1]), (ws[2], None, ys[2]), (ws[1], None, ys[3]), (ws[2], ws[0], ys[4])]), be.last_error()
        assert row_err(ys[0], oxref.gguf_decode(kind, raws[0], n_out, n_in, x, t)) < 1e-3
        assert np.array_equal(ys[1].view(np.uint32), oxref.silu_mul(ys[0], ys[3]).view(np.uint32))
        assert np.array_equal(ys[4].view(np.uint32), oxref.silu_mul(ys[2], ys[0]).view(np.uint32))
        alone = np.zeros((t, n_out), np.float32)
        assert be.matvec_rows(x, t, n_in, [(ws[2], None, alone)])
        assert np.array_equal(alone.view(np.uint32), ys[2].view(np.uint32))


def test_matvec_rows_of_full_size_pairs_keep_the_bits(be, oxref):
    """A call large enough for the shared launch's fat mapping (several K slices per workgroup, several runs per wave), with
    gate / up pairs in it: Llama-8B MLP shapes in Q8_0 and Q4_K, plain and paired. Every plain job gives the rows of a
    call of its own, every pair silu_mul of its two plain products, bit for bit."""
    from oxinfer_amd import synth
    gens = {8: synth.gguf_q8_0, 12: synth.gguf_q4_k}
    up_shape, down_shape = (14336, 4096), (4096, 14336)
    ws = {(kind, i): be.upload_gguf(kind, gens[kind](*up_shape, 20 + kind + i), *up_shape) for kind in gens for i in range(2)}
    for t in (1, 4):
        x = synth.activations(t, up_shape[1], 30 + t)
        names = [(kind, i) for kind in gens for i in range(2)]
        plain = {nm: np.zeros((t, up_shape[0]), np.float32) for nm in names}
        for nm in names:  # each alone
            assert be.matvec_rows(x, t, up_shape[1], [(ws[nm], None, plain[nm])]), be.last_error()
        together = {nm: np.zeros((t, up_shape[0]), np.float32) for nm in names}
        pairs = {kind: np.zeros((t, up_shape[0]), np.float32) for kind in gens}
        jobs = [(ws[nm], None, together[nm]) for nm in names] + [(ws[(kind, 0)], ws[(kind, 1)], pairs[kind]) for kind in gens]
        assert be.matvec_rows(x, t, up_shape[1], jobs), be.last_error()
        for nm in names:
            assert np.array_equal(together[nm].view(np.uint32), plain[nm].view(np.uint32)), (t, nm)
        for kind in gens:
            want = oxref.silu_mul(plain[(kind, 0)], plain[(kind, 1)])
            assert np.array_equal(pairs[kind].view(np.uint32), want.view(np.uint32)), (t, kind)
    # the long-K shape (K sliced across workgroups), paired
    wd = {(kind, i): be.upload_gguf(kind, gens[kind](*down_shape, 60 + kind + i), *down_shape) for kind in gens for i in range(2)}
    t = 2
    x = synth.activations(t, down_shape[1], 77)
    plain = {nm: np.zeros((t, down_shape[0]), np.float32) for nm in wd}
    for nm in wd:
        assert be.matvec_rows(x, t, down_shape[1], [(wd[nm], None, plain[nm])]), be.last_error()
    pairs = {kind: [np.zeros((t, down_shape[0]), np.float32) for _ in range(4)] for kind in gens}
    jobs = [(wd[(kind, 0)], wd[(kind, 1)], y) for kind in gens for y in pairs[kind]] + [(wd[nm], None, np.zeros((t, down_shape[0]), np.float32)) for nm in wd]
    assert be.matvec_rows(x, t, down_shape[1], jobs), be.last_error()
    for kind in gens:
        want = oxref.silu_mul(plain[(kind, 0)], plain[(kind, 1)])
        for y in pairs[kind]:
            assert np.array_equal(y.view(np.uint32), want.view(np.uint32)), kind
