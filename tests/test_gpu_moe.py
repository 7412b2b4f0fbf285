"""Routed-expert block on the GPU against oracle/moe.py, and the W8 expert
GEMV against the reference's own expert test pattern
(ollama-xdna/backend/test_experts.cpp:58-182)."""

import numpy as np
import pytest

from _util import announce, rel_l2
from oracle import bf16
from oracle.moe import moe_forward, route

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def moe_weights():
    from runtime.moe import synthetic_moe

    return synthetic_moe(seed=0)


@pytest.fixture(scope="module")
def block(moe_weights):
    from runtime.moe import MoEBlock

    router, gate_up, down = moe_weights
    b = MoEBlock(router, gate_up, down, top_k=6, shared=2, max_tokens=16)
    yield b
    b.close()


def _tie_gap(probs, k):
    """Gap between the k-th and (k+1)-th largest router probabilities."""
    s = np.sort(probs)[::-1]
    return float(s[k - 1] - s[k])


@pytest.mark.parametrize("tokens", [1, 2, 4, 8, 16])
def test_moe_block_matches_oracle(block, moe_weights, tokens):
    router, gate_up, down = moe_weights
    announce(f"moe block T={tokens}")
    rng = np.random.default_rng(100 + tokens)
    x = bf16.to_bits(rng.normal(0, 1, (tokens, 2048)).astype(np.float32))
    y, ids, w = block.forward(x)
    ref_y, ref_ids, ref_w = moe_forward(x, router, gate_up, down, top_k=6, shared=2)
    for t in range(tokens):
        _, _, probs = route(router, bf16.from_bits(x[t]), 6)
        if not np.array_equal(ids[t], ref_ids[t]):
            # only a float32 near-tie of the router may reorder or swap experts
            gaps = [_tie_gap(probs, k) for k in range(1, 7)]
            assert min(gaps) < 1e-6, (t, ids[t], ref_ids[t], gaps)
            continue
        np.testing.assert_allclose(w[t], ref_w[t], rtol=1e-5, atol=1e-7)
        err = rel_l2(bf16.from_bits(y[t]), bf16.from_bits(ref_y[t]))
        assert err <= 1e-2, (t, err)


def test_moe_block_beyond_16_tokens_matches_oracle(moe_weights):
    """24 tokens: groups of more than 16 rows (the shared experts), and the
    top-k in a launch of its own."""
    from runtime.moe import MoEBlock

    router, gate_up, down = moe_weights
    announce("moe block T=24")
    b = MoEBlock(router, gate_up, down, top_k=6, shared=2, max_tokens=32)
    try:
        rng = np.random.default_rng(124)
        x = bf16.to_bits(rng.normal(0, 1, (24, 2048)).astype(np.float32))
        y, ids, w = b.forward(x)
    finally:
        b.close()
    ref_y, ref_ids, ref_w = moe_forward(x, router, gate_up, down, top_k=6, shared=2)
    for t in range(24):
        if not np.array_equal(ids[t], ref_ids[t]):
            _, _, probs = route(router, bf16.from_bits(x[t]), 6)
            assert min(_tie_gap(probs, k) for k in range(1, 7)) < 1e-6, (t, ids[t], ref_ids[t])
            continue
        np.testing.assert_allclose(w[t], ref_w[t], rtol=1e-5, atol=1e-7)
        assert rel_l2(bf16.from_bits(y[t]), bf16.from_bits(ref_y[t])) <= 1e-2, t


def test_moe_experts_with_given_routing(block, moe_weights):
    """The MUL_MAT_ID form with caller ids equals the routed forward."""
    announce("moe experts with given ids")
    rng = np.random.default_rng(7)
    x = bf16.to_bits(rng.normal(0, 1, (5, 2048)).astype(np.float32))
    y, ids, w = block.forward(x)
    y2 = block.experts(x, ids, w)
    np.testing.assert_array_equal(y, y2)
    bad = ids.copy()
    bad[0, 0] = 64
    with pytest.raises(ValueError):
        block.experts(x, bad, w)


def test_moe_experts_repeated_ids_beyond_16_rows(block, moe_weights):
    """Caller ids may name one expert several times per token: 3 tokens x 6
    times expert 3 is 18 rows for one expert, more than one 16-row block;
    against the oracle's experts and combine (oracle/moe.py moe_forward's order)."""
    from oracle.moe import expert_forward

    router, gate_up, down = moe_weights
    announce("moe experts, one expert named 18 times")
    rng = np.random.default_rng(9)
    x = bf16.to_bits(rng.normal(0, 1, (3, 2048)).astype(np.float32))
    ids = np.full((3, 6), 3, dtype=np.int32)
    w = rng.uniform(0.05, 0.3, (3, 6)).astype(np.float32)
    y = block.experts(x, ids, w)
    for t in range(3):
        xt = bf16.from_bits(x[t])
        e3 = expert_forward(gate_up[3], down[3], xt)
        acc = np.zeros(2048, dtype=np.float32)
        for k in range(6):
            acc = acc + w[t, k] * e3
        for s_ in range(2):
            acc = acc + expert_forward(gate_up[64 + s_], down[64 + s_], xt)
        assert rel_l2(bf16.from_bits(y[t]), bf16.from_bits(bf16.to_bits(acc))) <= 1e-2, t


@pytest.mark.parametrize("tokens", [16, 17, 33, 65, 130, 256])
@pytest.mark.parametrize("shape", [(96, 32, 5, 0, 3), (64, 160, 64, 2, 6)])
def test_moe_row_groups_match_oracle(tokens, shape):
    """Groups of 1..64 rows (each row-block count of the expert slabs) and
    experts of more rows than one group, K of fewer and of more 32-column
    steps than waves, with and without shared experts; then the same routing
    given by the caller, with one token's experts all the same."""
    from oracle.moe import expert_forward
    from runtime.moe import MoEBlock, synthetic_moe

    H, I, E, S, K = shape
    announce(f"moe row groups T={tokens} {shape}")
    router, gate_up, down = synthetic_moe(dict(hidden=H, intermediate=I, experts=E, shared=S), seed=3, std=0.1)
    rng = np.random.default_rng(tokens)
    x = bf16.to_bits(rng.normal(0, 1, (tokens, H)).astype(np.float32))
    b = MoEBlock(router, gate_up, down, top_k=K, shared=S, max_tokens=256)
    try:
        y, ids, w = b.forward(x)
        ids2 = ids.copy()
        ids2[tokens // 2] = ids2[tokens // 2, 0]
        y2 = b.experts(x, ids2, w)
        y3 = b.experts(x, np.full_like(ids, ids[0, 0]), w) if tokens == 16 else None
    finally:
        b.close()
    ref_y, ref_ids, ref_w = moe_forward(x, router, gate_up, down, top_k=K, shared=S)
    for t in range(tokens):
        if not np.array_equal(ids[t], ref_ids[t]):
            _, _, probs = route(router, bf16.from_bits(x[t]), K)
            assert min(_tie_gap(probs, k) for k in range(1, K + 1)) < 1e-6, (t, ids[t], ref_ids[t])
            continue
        np.testing.assert_allclose(w[t], ref_w[t], rtol=1e-5, atol=1e-7)
        assert rel_l2(bf16.from_bits(y[t]), bf16.from_bits(ref_y[t])) <= 1e-2, t
    same = [t for t in range(tokens) if t != tokens // 2]
    np.testing.assert_array_equal(y2[same], y[same])

    def all_on(e, t):
        """Token t's output with every choice on expert e."""
        xt = bf16.from_bits(x[t])
        out = expert_forward(gate_up[e], down[e], xt)
        acc = np.zeros(H, dtype=np.float32)
        for k in range(K):
            acc = acc + w[t, k] * out
        for s in range(S):
            acc = acc + expert_forward(gate_up[E + s], down[E + s], xt)
        return bf16.from_bits(bf16.to_bits(acc))

    t = tokens // 2
    assert rel_l2(bf16.from_bits(y2[t]), all_on(ids2[t, 0], t)) <= 1e-2
    if y3 is not None:  # more than one group of one expert (96 rows of the second shape)
        for t in range(tokens):
            assert rel_l2(bf16.from_bits(y3[t]), all_on(ids[0, 0], t)) <= 1e-2, t


@pytest.mark.parametrize("tokens", [3, 20, 48, 150])
def test_moe_rows_longer_than_the_ring(tokens):
    """More K steps per wave than its ring holds, whole and partial last rounds,
    on one, two and four 16-row blocks, narrow and wide."""
    from runtime.moe import MoEBlock, synthetic_moe

    H, I, E, K = 2336, 2080, 2, 2
    announce(f"moe long rows T={tokens}")
    router, gate_up, down = synthetic_moe(dict(hidden=H, intermediate=I, experts=E, shared=0), seed=4)
    x = bf16.to_bits(np.random.default_rng(tokens).normal(0, 1, (tokens, H)).astype(np.float32))
    b = MoEBlock(router, gate_up, down, top_k=K, shared=0, max_tokens=256)
    try:
        y, ids, w = b.forward(x)
    finally:
        b.close()
    some = sorted({0, tokens // 2, tokens - 1})
    ref_y, _, ref_w = moe_forward(x[some], router, gate_up, down, top_k=K, shared=0)
    for i, t in enumerate(some):
        np.testing.assert_allclose(w[t], ref_w[i], rtol=1e-5, atol=1e-7)
        assert rel_l2(bf16.from_bits(y[t]), bf16.from_bits(ref_y[i])) <= 1e-2, t


@pytest.mark.parametrize("hidden,intermediate,tokens",
                         [(32768, 32800, 3), (32768, 32800, 40), ((1 << 23) + 32, 64, 130), (64, (1 << 24) + 32, 70)])
def test_moe_experts_of_more_than_2_gib(hk_lib, hidden, intermediate, tokens):
    """Expert matrices and token rows that no 32-bit size spans: gate/up of
    4 GiB per expert on few and many rows, 2 GiB of token rows (two passes), and
    of a group's intermediate rows.
    All zero but for the first and last hidden columns and intermediate rows, so
    the oracle runs on those alone."""
    import ctypes

    from oracle.moe import expert_forward
    from runtime import hip
    from runtime.moe import MoEDesc

    H, I, n = hidden, intermediate, 2  # one routed and one shared expert
    announce(f"moe H={H} I={I} T={tokens}")
    rng = np.random.default_rng(tokens)
    bits = lambda *shape: bf16.to_bits(rng.normal(0, 0.3, shape).astype(np.float32))  # noqa: E731
    columns, rows = (0, 32, H - 32), (0, 16, I - 16)  # two runs each: starts 0 and the last, their length between

    def zeros(count):
        b = hip.DeviceBuffer(2 * count)
        b.zero()
        return b

    def runs(spec):
        return [(spec[0], 0), (spec[2], spec[1])], spec[1]  # (start in the whole, start in the part), length

    def place(buf, first, line, part, lines, spec):
        """part's rows at the lines `lines` (each `line` long, from element `first`), in the runs of `spec`."""
        starts, length = runs(spec)
        for i, at in enumerate(lines):
            for big, small in starts:
                buf.write(part[i, small:small + length], 2 * (first + at * line + big))

    def ends(spec):
        starts, length = runs(spec)
        return [big + i for big, _ in starts for i in range(length)]

    x, gate_up, down = bits(tokens, 64), bits(n, 64, 64), bits(n, 64, 32)
    bufs = dict(x=zeros(tokens * H), gate_up=zeros(n * 2 * I * H), down=zeros(n * H * I), y=zeros(tokens * H),
                router=zeros(H))
    place(bufs["x"], 0, H, x, range(tokens), columns)
    for e in range(n):
        inter = ends(rows)
        place(bufs["gate_up"], e * 2 * I * H, H, gate_up[e], inter + [I + i for i in inter], columns)
        place(bufs["down"], e * H * I, I, down[e], ends(columns), rows)
    handle = ctypes.c_void_p()
    desc = MoEDesc(hidden=H, intermediate=I, experts=1, shared=1, top_k=1, max_tokens=tokens)
    try:
        hip.check(hk_lib.hk_moe_create(ctypes.byref(desc), bufs["router"].ptr, bufs["gate_up"].ptr, bufs["down"].ptr,
                                       ctypes.byref(handle)), "hk_moe_create")
        hip.check(hk_lib.hk_moe_forward(handle.value, bufs["x"].ptr, tokens, bufs["y"].ptr, None, None, None), "moe")
        hip.check(hk_lib.hk_stream_sync(None), "sync")
        starts, length = runs(columns)
        y = np.stack([np.concatenate([bufs["y"].read(np.uint16, length, 2 * (t * H + big)) for big, _ in starts])
                      for t in range(tokens)])
        middle = bufs["y"].read(np.uint16, H - 64, 2 * ((tokens - 1) * H + 32))
    finally:
        if handle.value:
            hk_lib.hk_moe_destroy(handle.value)
        for b in bufs.values():
            b.free()
    assert not middle.any()
    for t in range(tokens):
        ref = sum(expert_forward(gate_up[e], down[e], bf16.from_bits(x[t])) for e in range(n))
        assert rel_l2(bf16.from_bits(y[t]), bf16.from_bits(bf16.to_bits(ref))) <= 1e-2, t


def test_w8_expert_gemv_reference_pattern(hk_lib):
    """8 experts x 2048x2048 int8 with the reference test's pattern, scales and
    inputs; max error against the float-accumulated expectation < 0.03 (the
    reference's bound) and within one bf16 rounding."""
    from runtime import hip

    announce("w8 expert gemv, reference pattern")
    E, R, C = 8, 2048, 2048
    r = np.arange(R)[:, None]
    c = np.arange(C)[None, :]
    worst = 0.0
    out_buf = hip.DeviceBuffer(2 * R)
    for e in range(E):
        wq = (((e * 7 + r * 3 + c * 5) % 31) - 15).astype(np.int8)
        scale = (0.0005 * (1 + (np.arange(R) % 5))).astype(np.float32)
        x = bf16.to_bits(np.float32(0.002) * ((((e + np.arange(C)) % 17) - 8).astype(np.float32)))
        Q, S, X = (hip.DeviceBuffer.from_array(a) for a in (wq, scale, x))
        hip.check(hk_lib.hk_gemv_w8(Q.ptr, S.ptr, X.ptr, None, None, out_buf.ptr, None, R, C, None), "w8")
        hip.check(hk_lib.hk_stream_sync(None), "sync")
        got = bf16.from_bits(out_buf.read(np.uint16, R))
        expected = (wq.astype(np.float32) @ bf16.from_bits(x)) * scale
        worst = max(worst, float(np.abs(got - expected).max()))
        # a float32 sum in another order may land on the other side of a
        # bf16 rounding boundary: one bf16 step
        ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(expected), 2.0**-126))) - 7)
        assert np.all(np.abs(got - expected) <= ulp * 1.0001 + 1e-6)
    assert worst < 0.03
