"""Small-M products (speculative-verify / prefill rows) vs M independent rows."""
import numpy as np
import pytest

from gpu_util import act_host, int_dot_tol, say, to_dev, to_host
from test_oracle import random_blocks

pytestmark = pytest.mark.gpu

_cache = {}

CASES = [  # type, rows, K, M, layout
    ("Q4_K", 6144, 5120, 1, 1), ("Q4_K", 6144, 5120, 2, 1), ("Q4_K", 6144, 5120, 4, 1),
    ("Q4_K", 6144, 5120, 8, 1), ("Q4_K", 6144, 5120, 16, 1), ("Q4_K", 6144, 5120, 23, 0),
    ("Q4_K", 40, 512, 5, 0), ("Q4_K", 40, 512, 64, 1),
    ("Q6_K", 5120, 17408, 16, 1), ("Q6_K", 5120, 17408, 3, 0), ("Q6_K", 24, 768, 9, 1),
    ("Q8_0", 2048, 6144, 16, 1), ("Q8_0", 2048, 6144, 2, 0), ("Q8_0", 13, 160, 7, 1),
    # few tokens: M = 2 on the GEMV-structured kernel (TILED Q4_K / Q5_K: on
    # MFMA with direct weight operands), M = 3 and 4 on MFMA (padding tokens,
    # partial 8-row tiles), each type
    ("Q6_K", 5120, 17408, 2, 1), ("Q6_K", 24, 768, 4, 1), ("Q4_K", 40, 512, 3, 1), ("Q8_0", 13, 160, 3, 1),
    ("Q8_0", 2048, 6144, 4, 1),
    # Q5_K on each path: few-token GEMV, MFMA, GGUF VALU
    ("Q5_K", 6144, 5120, 2, 1), ("Q5_K", 6144, 5120, 16, 1), ("Q5_K", 40, 512, 9, 1), ("Q5_K", 40, 512, 3, 0),
    # IQ4_XS likewise
    ("IQ4_XS", 6144, 5120, 2, 1), ("IQ4_XS", 6144, 5120, 16, 1), ("IQ4_XS", 40, 512, 9, 1),
    ("IQ4_XS", 40, 512, 3, 0),
    # MFMA with two 16-row sets per tile (M <= 8 and >= 128 sets of 32 rows):
    # a partial last set (8200 rows), a partial Q8_0 unit (K = 160), every
    # type; 24 tokens on the wide kernel
    ("Q4_K", 8200, 512, 5, 1), ("Q4_K", 8192, 512, 8, 1), ("Q4_K", 8192, 512, 24, 1),
    ("Q6_K", 8200, 768, 7, 1), ("Q8_0", 8200, 160, 6, 1), ("Q5_K", 8192, 512, 8, 1),
    ("IQ4_XS", 8200, 512, 6, 1),
    # gate-sized rows at M = 3 (two sets per tile), the down shape at M = 12
    # (padding tokens in a 16-token launch), 17 tokens on the wide kernel
    ("Q4_K", 17408, 5120, 3, 1), ("Q6_K", 5120, 17408, 12, 1), ("Q4_K", 8192, 512, 17, 1),
    # few tokens with balanced tiling on 256 CUs (rows under 40 units) on the
    # GEMV-structured kernel (Q6_K), and the same shapes on MFMA with direct
    # operands (Q4_K): o, a ragged last tile
    ("Q4_K", 5120, 6144, 2, 1), ("Q6_K", 4100, 2048, 2, 1), ("Q4_K", 6141, 2048, 2, 1),
    # direct weight operands at M = 2: a single partial tile, a partial last
    # two-set tile, and gate-sized rows (544 workgroups: K over 4 waves)
    ("Q4_K", 13, 256, 2, 1), ("Q5_K", 8200, 512, 2, 1), ("Q4_K", 17408, 1024, 2, 1),
    # resident activation rows (16-token launches with >= 4 row sets per CU:
    # 1025 sets of 16 rows on 256 CUs), every type, a partial last set, a
    # partial Q8_0 unit (K = 1056); 25 and 32 tokens on the wide kernel
    ("Q4_K", 16390, 1024, 16, 1), ("Q6_K", 16390, 1024, 16, 1), ("Q8_0", 16390, 1056, 16, 1),
    ("Q5_K", 16390, 1024, 25, 1), ("IQ4_XS", 16390, 1024, 32, 1),
    # two row sets per tile over 1025 sets of 32 rows (a last set of 8 rows),
    # every type, padding tokens
    ("Q4_K", 32776, 512, 8, 1), ("Q6_K", 32776, 768, 5, 1), ("Q8_0", 32776, 160, 7, 1),
    ("Q5_K", 32776, 512, 3, 1), ("IQ4_XS", 32776, 512, 8, 1),
    # GGUF-layout K-quants on the MFMA kernel, staged from the row blocks:
    # from M = 2, two-set tiles with a partial last set, 16-token resident
    # launches (Q6_K: the per-unit kernel), 16 + 3 tokens (257 sets) and padding
    # tokens, 25 tokens on the wide kernel; Q6_K rows of an
    # odd block count (K = 768, 2304: every other row starts 2 bytes past a
    # multiple of 4) and the down shape
    ("Q4_K", 6144, 5120, 2, 0), ("Q4_K", 8200, 512, 6, 0), ("Q4_K", 16390, 1024, 16, 0), ("Q4_K", 4100, 1024, 19, 0),
    ("Q5_K", 6144, 5120, 2, 0), ("Q5_K", 8200, 512, 8, 0), ("Q5_K", 16390, 1024, 25, 0),
    ("Q6_K", 24, 768, 2, 0), ("Q6_K", 8200, 768, 7, 0), ("Q6_K", 16390, 1024, 16, 0), ("Q6_K", 1030, 2304, 11, 0),
    ("Q6_K", 5120, 17408, 16, 0), ("Q6_K", 33, 2304, 4, 0),
    # GGUF-layout weights at M = 2 on the few-token kernel: o's shape (balanced
    # over one workgroup per CU), IQ4_XS and Q8_0 (its 34-byte blocks)
    ("Q4_K", 5120, 6144, 2, 0), ("IQ4_XS", 40, 512, 2, 0), ("Q8_0", 13, 160, 2, 0),
]


@pytest.mark.parametrize("type_name,rc,k,M,layout", CASES)
def test_matmul_vs_oracle(m27q, ora, dev, type_name, rc, k, M, layout):
    import torch
    t = getattr(m27q, type_name)
    rb = k // m27q.BLOCK_ELEMS[t]
    key = (type_name, rc, k)
    if key not in _cache:
        _cache[key] = ora.synth_weights(t, rc, k, seed=40)
    wb = _cache[key]
    w = m27q.Weight.upload(wb.reshape(-1), t, rb, rc, layout, dev)
    X = np.random.default_rng(M).standard_normal((M, k)).astype(np.float32)
    act = m27q.Act(M, k, dev)
    m27q.quant_act(to_dev(X, dev), act)
    res = np.random.default_rng(M + 1).standard_normal((M, rc)).astype(np.float32)
    Y = torch.empty((M, rc), dtype=torch.float32, device=dev)
    say("matmul", type_name, rc, k, M, layout)
    m27q.matmul_q8(w, act, Y, residual=to_dev(res, dev))
    got = to_host(Y).astype(np.float64) - res
    q, d, s = act_host(m27q, act)
    for m in range(M):
        want, nrm = ora.gemv_act(t, wb, rb, rc, q[m], d[m], s[m])
        assert (np.abs(got[m] - want) <= int_dot_tol(nrm) + 1e-6 * np.abs(res[m])).all(), m


@pytest.mark.parametrize("M", [2, 5, 16, 19])
def test_matmul_multi_vs_oracle(m27q, ora, dev, M):
    """q/k/v-shaped weights on one activation in one launch, each against the
    integer-dot oracle (row subsets), across the 16-token launch boundary (M = 19:
    a launch of 16 tokens and one of 3)."""
    import torch
    k, shapes = 5120, [6144, 1024, 1024]
    wbs = [ora.synth_weights(m27q.Q4_K, rc, k, seed=60 + i) for i, rc in enumerate(shapes)]
    ws = [m27q.Weight.upload(wb.reshape(-1), m27q.Q4_K, 20, rc, m27q.TILED, dev) for wb, rc in zip(wbs, shapes)]
    X = np.random.default_rng(M + 7).standard_normal((M, k)).astype(np.float32)
    act = m27q.Act(M, k, dev)
    m27q.quant_act(to_dev(X, dev), act)
    Ys = [torch.empty((M, rc), dtype=torch.float32, device=dev) for rc in shapes]
    say("matmul multi", M)
    m27q.matmul_q8_multi(ws, act, Ys)
    q, d, s = act_host(m27q, act)
    for wb, rc, Y in zip(wbs, shapes, Ys):
        got = to_host(Y).astype(np.float64)
        for m in sorted({0, M // 2, M - 1}):
            want, nrm = ora.gemv_act(m27q.Q4_K, wb, 20, rc, q[m], d[m], s[m])
            assert (np.abs(got[m] - want) <= int_dot_tol(nrm)).all(), (rc, m)


@pytest.mark.parametrize("M,rows", [(16, 8200), (32, 8200), (7, 16400)])
def test_matmul_multi_resident_vs_oracle(m27q, ora, dev, M, rows):
    """Two weights of one K in one launch over 1026 row sets: at M = 16 the
    resident-activation kernel (the second matrix's sets following the first's
    in the workgroups' runs), at M = 32 the wide kernel, at M = 7 the two-set
    per-unit kernel; each against the integer-dot oracle."""
    import torch
    k, shapes = 1024, [rows, rows]
    wbs = [ora.synth_weights(m27q.Q4_K, rc, k, seed=70 + i) for i, rc in enumerate(shapes)]
    ws = [m27q.Weight.upload(wb.reshape(-1), m27q.Q4_K, 4, rc, m27q.TILED, dev) for wb, rc in zip(wbs, shapes)]
    X = np.random.default_rng(M + 9).standard_normal((M, k)).astype(np.float32)
    act = m27q.Act(M, k, dev)
    m27q.quant_act(to_dev(X, dev), act)
    Ys = [torch.empty((M, rc), dtype=torch.float32, device=dev) for rc in shapes]
    say("matmul multi resident", M)
    m27q.matmul_q8_multi(ws, act, Ys)
    q, d, s = act_host(m27q, act)
    for wb, rc, Y in zip(wbs, shapes, Ys):
        got = to_host(Y).astype(np.float64)
        for m in range(M):
            want, nrm = ora.gemv_act(m27q.Q4_K, wb, 4, rc, q[m], d[m], s[m])
            assert (np.abs(got[m] - want) <= int_dot_tol(nrm)).all(), (rc, m)


@pytest.mark.parametrize("M", [2, 9, 16])
def test_matmul_multi_gguf_vs_oracle(m27q, ora, dev, M):
    """GGUF-layout weights through the multi entry point: Q4_K q/k/v-shaped
    weights in one MFMA launch, then a mixed group (Q6_K on the MFMA kernel,
    Q8_0 on the wide one; M = 2 on the few-token kernel) on the same activation;
    every token row of each output against the integer-dot oracle."""
    import torch
    k = 1536
    spec = [("Q4_K", 6144, 80), ("Q4_K", 1024, 81), ("Q4_K", 1024, 82)]
    mixed = [("Q6_K", 1030, 83), ("Q8_0", 515, 84)]
    X = np.random.default_rng(M + 11).standard_normal((M, k)).astype(np.float32)
    act = m27q.Act(M, k, dev)
    m27q.quant_act(to_dev(X, dev), act)
    q, d, s = act_host(m27q, act)
    for group in (spec, mixed):
        wbs, ws, rbs = [], [], []
        for name, rc, seed in group:
            t = getattr(m27q, name)
            rb = k // m27q.BLOCK_ELEMS[t]
            wb = ora.synth_weights(t, rc, k, seed=seed)
            wbs.append(wb)
            rbs.append(rb)
            ws.append(m27q.Weight.upload(wb.reshape(-1), t, rb, rc, m27q.GGUF, dev))
        Ys = [torch.empty((M, rc), dtype=torch.float32, device=dev) for _, rc, _ in group]
        say("matmul multi gguf", M, [g[0] for g in group])
        m27q.matmul_q8_multi(ws, act, Ys)
        for (name, rc, _), wb, rb, Y in zip(group, wbs, rbs, Ys):
            got = to_host(Y).astype(np.float64)
            for m in range(M):
                want, nrm = ora.gemv_act(getattr(m27q, name), wb, rb, rc, q[m], d[m], s[m])
                assert (np.abs(got[m] - want) <= int_dot_tol(nrm)).all(), (name, rc, m)


@pytest.mark.parametrize("type_name,rc,k", [("Q6_K", 1030, 2304), ("Q6_K", 8200, 768), ("Q6_K", 4098, 6144),
                                            ("Q8_0", 515, 1056)])
def test_gguf_two_byte_aligned_base(m27q, ora, dev, type_name, rc, k):
    """GGUF Q6_K and Q8_0 weights need only 2-byte alignment: the matrix placed
    2 bytes past a multiple of 4 (a view into a larger buffer).  The M = 1
    products (quantized and fp32 x; one- and two-tile waves read Q6_K's fields
    as shifted dwords or halfwords) and the small-M products (Q6_K: the MFMA
    kernel with one- and two-set tiles, whose staging reads dwords from the
    4-aligned address below each chunk; Q8_0: the wide kernel), every token
    row against the integer-dot oracle."""
    import torch
    t = getattr(m27q, type_name)
    rb = k // m27q.BLOCK_ELEMS[t]
    wb = ora.synth_weights(t, rc, k, seed=90)
    raw = torch.from_numpy(wb.reshape(-1).copy()).to(dev)
    buf = torch.zeros(raw.numel() + 2, dtype=torch.uint8, device=dev)
    buf[2:] = raw
    w = m27q.Weight(buf[2:], t, rb, rc, m27q.GGUF)
    assert w.data.data_ptr() % 4 == 2
    rng = np.random.default_rng(91)
    for M in (1, 2, 7, 16):
        X = rng.standard_normal((M, k)).astype(np.float32)
        act = m27q.Act(M, k, dev)
        m27q.quant_act(to_dev(X, dev), act)
        q, d, s = act_host(m27q, act)
        Y = torch.empty((M, rc), dtype=torch.float32, device=dev)
        say("gguf 2-byte base", type_name, rc, k, M)
        m27q.matmul_q8(w, act, Y)
        got = to_host(Y).astype(np.float64)
        for m in range(M):
            want, nrm = ora.gemv_act(t, wb, rb, rc, q[m], d[m], s[m])
            assert (np.abs(got[m] - want) <= int_dot_tol(nrm)).all(), (M, m)
        if M == 1:
            y = torch.empty(rc, dtype=torch.float32, device=dev)
            m27q.matvec(w, to_dev(X[0], dev), y)
            qf, df, sf = ora.quant_act(X[0])
            want, nrm = ora.gemv_act(t, wb, rb, rc, qf, df, sf)
            assert (np.abs(to_host(y).astype(np.float64) - want) <= int_dot_tol(nrm)).all(), "fp32 x"


WIDE = [  # type, rows, K, M, layout: the wide kernel's launch shapes on 256 CUs (16-row sets per CU)
    # up to one set per CU (K over 8 waves): one partial set, K of one unit
    # (seven waves without work), a unit count the slices do not divide
    ("Q4_K", 13, 256, 17, 1), ("Q5_K", 40, 2304, 33, 0), ("Q6_K", 40, 2304, 64, 1), ("Q6_K", 13, 256, 49, 0),
    ("IQ4_XS", 40, 512, 64, 1), ("Q8_0", 13, 32, 17, 1), ("Q8_0", 40, 1056, 64, 1), ("Q8_0", 13, 160, 9, 0),
    # ... of 5 and 8 rows
    ("Q8_0", 13, 384, 5, 0), ("IQ4_XS", 13, 1280, 5, 0), ("Q8_0", 4095, 416, 8, 0),
    # two row waves of at most one set: an odd set count (257: a wave without a
    # set), a partial last 8-row tile and set
    ("Q4_K", 4100, 1024, 33, 1), ("Q4_K", 4100, 256, 64, 0), ("Q5_K", 4100, 512, 48, 1), ("Q6_K", 4100, 768, 64, 0),
    ("Q6_K", 8185, 512, 64, 1), ("IQ4_XS", 4100, 512, 37, 0), ("Q8_0", 4100, 160, 64, 0), ("Q8_0", 4100, 288, 33, 1),
    # two row waves of up to three sets (2.0 to 6 sets per CU)
    ("Q4_K", 8210, 512, 64, 1), ("Q5_K", 12301, 256, 17, 0), ("Q6_K", 24570, 256, 64, 1), ("Q8_0", 12301, 96, 47, 0),
    ("IQ4_XS", 8210, 512, 64, 0),
    # four row waves of up to three sets: just above 6 sets per CU, two rounds
    ("Q4_K", 24600, 512, 64, 1), ("Q5_K", 50001, 256, 33, 1), ("Q6_K", 24600, 256, 33, 0), ("Q8_0", 24600, 160, 64, 1),
    ("IQ4_XS", 24600, 256, 20, 0), ("Q4_K", 24600, 256, 17, 0),
    # 9 and 16 rows on two row waves of up to three sets (521 and 770 sets) and on
    # four (1538), partial last sets
    ("Q8_0", 8330, 416, 9, 0), ("Q8_0", 12310, 1024, 16, 0), ("Q8_0", 24605, 2560, 9, 0),
    ("IQ4_XS", 8330, 512, 16, 0), ("IQ4_XS", 12310, 1280, 9, 0), ("IQ4_XS", 24605, 1280, 16, 0),
]
# 5 rows of a short K, which the VALU kernel keeps
VALU_SHORT = [("Q8_0", 13, 32, 5, 0), ("IQ4_XS", 13, 256, 5, 0)]
# 17 to 32 rows on the MFMA kernel (257 and 385 sets; a launch of 16 rows, then one
# of up to 8 rows on two-set tiles or of more on one-set ones), partial last sets;
# 3075 sets, past 12 per CU: the resident kernel, then one row
TWO_LAUNCHES = [
    ("Q4_K", 4100, 1024, 17, 1), ("Q4_K", 4100, 1024, 24, 1), ("Q4_K", 4100, 1024, 32, 1),
    ("Q5_K", 4100, 512, 17, 1), ("Q5_K", 4100, 512, 24, 1), ("Q5_K", 4100, 512, 32, 1), ("Q5_K", 4100, 512, 24, 0),
    ("Q6_K", 4100, 768, 17, 1), ("Q6_K", 4100, 768, 24, 1), ("Q6_K", 4100, 768, 32, 1),
    ("Q6_K", 4100, 768, 17, 0), ("Q6_K", 6150, 768, 32, 0), ("Q4_K", 4100, 512, 32, 0),
    ("Q8_0", 4100, 1056, 17, 1), ("Q8_0", 4100, 1056, 24, 1), ("Q8_0", 4100, 1056, 32, 1),
    ("IQ4_XS", 4100, 512, 17, 1), ("IQ4_XS", 6150, 512, 24, 1), ("IQ4_XS", 6150, 512, 32, 1),
    ("Q8_0", 49195, 544, 17, 1),
]


@pytest.mark.parametrize("type_name,rc,k,M,layout", WIDE + VALU_SHORT + TWO_LAUNCHES)
def test_wide_vs_oracle(m27q, ora, dev, type_name, rc, k, M, layout):
    """One launch of up to 64 rows, or the launches of 16 that it replaces
    elsewhere (the first, last and tile-edge tokens, with a residual) against
    the integer-dot oracle.  The scaled integer sums are
    exact, so what differs is the order of the fp32 sums over groups and
    blocks: the bar of every product (int_dot_tol)."""
    import torch
    t = getattr(m27q, type_name)
    rb = k // m27q.BLOCK_ELEMS[t]
    wb = ora.synth_weights(t, rc, k, seed=41)
    w = m27q.Weight.upload(wb.reshape(-1), t, rb, rc, layout, dev)
    X = np.random.default_rng(M).standard_normal((M, k)).astype(np.float32)
    X[:, : k // 2] *= 1000.0  # groups of very different scale
    act = m27q.Act(M, k, dev)
    m27q.quant_act(to_dev(X, dev), act)
    res = np.random.default_rng(M + 1).standard_normal((M, rc)).astype(np.float32)
    Y = torch.full((M + 1, rc), 7.0, dtype=torch.float32, device=dev)
    say("wide", type_name, rc, k, M, layout)
    m27q.matmul_q8(w, act, Y[:M], residual=to_dev(res, dev))
    got = to_host(Y).astype(np.float64)
    assert (got[M] == 7.0).all()  # nothing written past the rows
    q, d, s = act_host(m27q, act)
    for m in sorted({0, min(15, M - 1), max(0, M // 16 * 16 - 1), min(M - 1, M // 16 * 16), M - 1}):
        want, nrm = ora.gemv_act(t, wb, rb, rc, q[m], d[m], s[m])
        assert (np.abs(got[m] - res[m] - want) <= int_dot_tol(nrm) + 1e-6 * np.abs(res[m])).all(), m


@pytest.mark.parametrize("shapes,M", [((6144, 1024, 1024), 64), ((100, 17, 3000, 2000), 33), ((9000, 9000, 9000), 48)])
def test_wide_multi_vs_oracle(m27q, ora, dev, shapes, M):
    """Several weights in one wide launch: workgroups whose sets belong to
    different weights, partial last sets in the middle of the run."""
    import torch
    k = 768
    for name in ("Q4_K", "Q6_K"):
        t = getattr(m27q, name)
        wbs = [ora.synth_weights(t, rc, k, seed=70 + i) for i, rc in enumerate(shapes)]
        ws = [m27q.Weight.upload(wb.reshape(-1), t, 3, rc, m27q.TILED, dev) for wb, rc in zip(wbs, shapes)]
        X = np.random.default_rng(M + 7).standard_normal((M, k)).astype(np.float32)
        act = m27q.Act(M, k, dev)
        m27q.quant_act(to_dev(X, dev), act)
        Ys = [torch.empty((M, rc), dtype=torch.float32, device=dev) for rc in shapes]
        say("wide multi", name, shapes, M)
        m27q.matmul_q8_multi(ws, act, Ys)
        q, d, s = act_host(m27q, act)
        for wb, rc, Y in zip(wbs, shapes, Ys):
            got = to_host(Y).astype(np.float64)
            for m in (0, M // 2, M - 1):
                want, nrm = ora.gemv_act(t, wb, 3, rc, q[m], d[m], s[m])
                assert (np.abs(got[m] - want) <= int_dot_tol(nrm)).all(), (name, rc, m)


@pytest.mark.parametrize("type_name,rc,k", [("Q6_K", 1030, 2304), ("Q6_K", 8210, 768), ("Q8_0", 515, 1056)])
def test_wide_two_byte_aligned_base(m27q, ora, dev, type_name, rc, k):
    """GGUF Q6_K / Q8_0 weights 2 bytes past a multiple of 4 on the wide kernel."""
    import torch
    t = getattr(m27q, type_name)
    rb = k // m27q.BLOCK_ELEMS[t]
    wb = ora.synth_weights(t, rc, k, seed=92)
    raw = torch.from_numpy(wb.reshape(-1).copy()).to(dev)
    buf = torch.zeros(raw.numel() + 2, dtype=torch.uint8, device=dev)
    buf[2:] = raw
    w = m27q.Weight(buf[2:], t, rb, rc, m27q.GGUF)
    M = 40
    act = m27q.Act(M, k, dev)
    m27q.quant_act(to_dev(np.random.default_rng(3).standard_normal((M, k)).astype(np.float32), dev), act)
    q, d, s = act_host(m27q, act)
    Y = torch.empty((M, rc), dtype=torch.float32, device=dev)
    say("wide 2-byte base", type_name, rc, k)
    m27q.matmul_q8(w, act, Y)
    got = to_host(Y).astype(np.float64)
    for m in (0, 17, M - 1):
        want, nrm = ora.gemv_act(t, wb, rb, rc, q[m], d[m], s[m])
        assert (np.abs(got[m] - want) <= int_dot_tol(nrm)).all(), m


@pytest.mark.parametrize("type_name,rc,M,layout,big", [
    ("Q4_K", 100, 20, 1, 1e36), ("Q4_K", 4200, 40, 0, 1e36), ("Q5_K", 100, 33, 0, 1e36), ("Q5_K", 4200, 64, 1, 1e36),
    ("Q6_K", 4200, 40, 1, 1e33), ("Q6_K", 100, 20, 0, 1e33), ("Q8_0", 4200, 40, 1, 1e37), ("IQ4_XS", 4200, 40, 1, 1e37)])
def test_wide_extreme_rows(m27q, ora, dev, type_name, rc, M, layout, big):
    """One activation row at the ends of the float range among ordinary ones:
    a row of magnitude `big` (the largest power of ten whose sums every other
    kernel keeps finite) and one of 1e-36 against the oracle, NaN values (code
    0) likewise, and a row with an infinity (NaN); the other rows' bits stay."""
    import torch
    t, k, r = getattr(m27q, type_name), 512, 7
    rb = k // m27q.BLOCK_ELEMS[t]
    wb = ora.synth_weights(t, rc, k, seed=3)
    w = m27q.Weight.upload(wb.reshape(-1), t, rb, rc, layout, dev)
    X0 = np.random.default_rng(5).standard_normal((M, k)).astype(np.float32)

    def product(X):
        act = m27q.Act(M, k, dev)
        m27q.quant_act(to_dev(X, dev), act)
        Y = torch.empty((M, rc), dtype=torch.float32, device=dev)
        m27q.matmul_q8(w, act, Y)
        return to_host(Y), [a[r] for a in act_host(m27q, act)]

    base, _ = product(X0)
    for name in ("big", "small", "nan", "inf"):
        X = X0.copy()
        if name == "nan":
            X[r, 3] = np.nan
            X[r, 32:64] = np.nan
        elif name == "inf":
            X[r, 3] = -np.inf
        else:
            X[r] = (X[r].astype(np.float64) * (big if name == "big" else 1e-36)).astype(np.float32)
        say("wide extreme", type_name, rc, M, layout, name)
        Y, (q, d, s) = product(X)
        assert np.array_equal(np.delete(Y, r, 0).view(np.uint32), np.delete(base, r, 0).view(np.uint32)), name
        if name == "inf":
            assert np.isnan(Y[r]).all()
            continue
        want, nrm = ora.gemv_act(t, wb, rb, rc, q, d, s)
        # 1e-36: every product and sum is also rounded to a multiple of 2^-149 (of
        # Q4_K / Q5_K's sums, kept 2^-10 down, 2^-139); Q8_0 / IQ4_XS round the
        # scales' product so before it meets a 12-bit sum
        tiny = k * 2.0 ** -149 * (2.0 ** 12 if type_name in ("Q8_0", "IQ4_XS") else 1024.0)
        assert (np.abs(Y[r].astype(np.float64) - want) <= 1e-6 * nrm + (tiny if name == "small" else 0)).all(), name


@pytest.mark.parametrize("type_name,rc,k,M", [
    ("Q8_0", 12401, 160, 9), ("Q8_0", 20003, 992, 16), ("IQ4_XS", 12401, 256, 16), ("IQ4_XS", 13000, 768, 11),
    ("Q8_0", 82001, 64, 17), ("Q8_0", 82001, 32, 24), ("IQ4_XS", 82001, 256, 20)])
def test_gguf_valu_16_rows(m27q, ora, dev, type_name, rc, k, M):
    """GGUF Q8_0 / IQ4_XS on many sets: launches of up to 16 rows of the VALU
    kernel (one or two units of K, ragged Q8_0 units, a second launch of 1, 4
    and 8 rows), every row with a residual against the oracle."""
    import torch
    t = getattr(m27q, type_name)
    rb = k // m27q.BLOCK_ELEMS[t]
    wb = ora.synth_weights(t, rc, k, seed=43)
    w = m27q.Weight.upload(wb.reshape(-1), t, rb, rc, m27q.GGUF, dev)
    act = m27q.Act(M, k, dev)
    m27q.quant_act(to_dev(np.random.default_rng(M).standard_normal((M, k)).astype(np.float32), dev), act)
    res = np.random.default_rng(M + 1).standard_normal((M, rc)).astype(np.float32)
    Y = torch.full((M + 1, rc), 7.0, dtype=torch.float32, device=dev)
    say("gguf valu", type_name, rc, k, M)
    m27q.matmul_q8(w, act, Y[:M], residual=to_dev(res, dev))
    got = to_host(Y).astype(np.float64)
    assert (got[M] == 7.0).all()
    q, d, s = act_host(m27q, act)
    for m in range(M):
        want, nrm = ora.gemv_act(t, wb, rb, rc, q[m], d[m], s[m])
        assert (np.abs(got[m] - res[m] - want) <= int_dot_tol(nrm) + 1e-6 * np.abs(res[m])).all(), m


def test_resident_second_launch(m27q, ora, dev):
    """32 rows in two launches of the resident-activation kernel: IQ4_XS, more
    than 12 sets per CU and a long K (random bytes: 194 MB of weights)."""
    import torch
    rc, k, M = 49200, 7424, 32
    rb = k // 256
    wb = random_blocks(ora, ora.IQ4_XS, rb * rc, np.random.default_rng(12))
    w = m27q.Weight.upload(wb.reshape(-1), m27q.IQ4_XS, rb, rc, m27q.TILED, dev)
    act = m27q.Act(M, k, dev)
    m27q.quant_act(to_dev(np.random.default_rng(13).standard_normal((M, k)).astype(np.float32), dev), act)
    Y = torch.empty((M, rc), dtype=torch.float32, device=dev)
    say("resident twice", rc, k, M)
    m27q.matmul_q8(w, act, Y)
    got = to_host(Y).astype(np.float64)
    q, d, s = act_host(m27q, act)
    for m in (0, 15, 16, 31):
        want, nrm = ora.gemv_act(ora.IQ4_XS, wb, rb, rc, q[m], d[m], s[m])
        assert (np.abs(got[m] - want) <= int_dot_tol(nrm)).all(), m


@pytest.mark.parametrize("type_name,layout", [(t, lay) for t in ("Q4_K", "Q5_K", "Q6_K", "Q8_0", "IQ4_XS") for lay in (0, 1)])
@pytest.mark.parametrize("rc,M", [(100, 17), (4100, 33), (8210, 64), (24600, 40)])
def test_wide_exact_integers(m27q, ora, dev, type_name, layout, rc, M):
    """Weights of block scale 1 (scales, mins and codes at their extremes among
    random ones) times codes with one power-of-two scale: every product and sum
    is a multiple of it below 2^24, so the results are exact, on each launch
    shape.  A lost bit of an operand (Q6_K's second fp16 value, a min term's
    third part) shows."""
    import torch
    t, k = getattr(m27q, type_name), 512
    rb = k // m27q.BLOCK_ELEMS[t]
    rng = np.random.default_rng(rc + M)
    b = rng.integers(0, 256, size=(rc * rb, ora.TYPE_SIZE[t]), dtype=np.uint8)
    one = np.frombuffer(np.float16(1).tobytes(), np.uint8)
    b[rng.random(b.shape) < 0.2] = 0x80 if type_name == "Q6_K" else 0xff  # Q6_K: scale -128 ...
    b[rng.random(b.shape) < 0.2] = 0x00                                   # ... and code -32
    off = 208 if type_name == "Q6_K" else 0
    b[:, off:off + 2] = one
    if type_name in ("Q4_K", "Q5_K"):
        b[:, 2:4] = one
    wb = b.reshape(rc, -1)
    w = m27q.Weight.upload(wb.reshape(-1), t, rb, rc, layout, dev)
    # two codes per group, one of them +-127 (so that the group's scale is 2^-3);
    # 16 groups x 2 x 127 x 4096 = 16,646,144 < 2^24
    X = np.zeros((M, k), np.float32)
    for m in range(M):
        for g in range(0, k, 32):
            i, j = rng.choice(32, 2, replace=False)
            X[m, g + i], X[m, g + j] = rng.choice([-127, 127]), rng.integers(-127, 128)
    act = m27q.Act(M, k, dev)
    m27q.quant_act(to_dev(X / 8, dev), act)
    q, d, s = act_host(m27q, act)
    assert np.array_equal(q, X) and (d == 0.125).all()
    Y = torch.empty((M, rc), dtype=torch.float32, device=dev)
    say("wide exact", type_name, layout, rc, M)
    m27q.matmul_q8(w, act, Y)
    # whole numbers up to 2^24: exact in a float64 product
    want = X.astype(np.float64) @ ora.dequant(t, wb, rb, rc).astype(np.float64).T / 8
    assert np.array_equal(to_host(Y).astype(np.float64), want)
