"""The M > 1 products of dequantised weights on the f32 matrix cores
(mm_f32.hip) against the oracle's a.dot order, bit for bit: int4 and q4a
linears and f16 / q4a expert matrices at the edges of the tiles (16 / 32 / 64
rows and columns), of the 32-long chunks and the 256-long blocks of k, for
groups of a multiple of 32, of 16 and of neither, and non-finite values."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SHAPES = [(2, 32, 1), (15, 64, 16), (16, 256, 17), (17, 288, 33), (31, 224, 64), (33, 512, 65), (48, 2304, 130),
          (64, 768, 63), (65, 544, 129), (129, 256, 300), (300, 320, 257), (3, 4608, 500), (70, 9216, 40),
          (520, 64, 700)]
RAGGED = [(2, 1, 3), (5, 31, 7), (17, 33, 40), (40, 255, 66), (64, 257, 65), (33, 1001, 129), (9, 2310, 31),
          (130, 790, 200)]


def same(got, ref):
    bad = np.argwhere(got.view(np.uint32) != ref.view(np.uint32))
    assert len(bad) == 0, (len(bad), bad[:4].tolist())


def packed_weight(rng, n, k, g):
    q = rng.integers(0, 256, (n, (k + 1) // 2), dtype=np.uint8)
    if k % 2:
        q[:, -1] &= 15
    s = rng.uniform(2e-3, 9e-3, (n, (k + g - 1) // g)).astype(np.float16)
    return q, s, (-7.5 * s.astype(np.float32)).astype(np.float16)


@pytest.mark.parametrize("g", [32, 64, 48, 16, 13])
@pytest.mark.parametrize("m,k,n", SHAPES + RAGGED)
def test_int4_and_q4a_in_a_dot_order(ctx, m, k, n, g):
    rng = np.random.default_rng(m * 31 + k * 7 + n + g)
    a = rng.standard_normal((m, k), dtype=np.float32)
    q, s, mn = packed_weight(rng, n, k, g)
    same(ctx.upload_i4(q, s, k, g).mm_exact(a), oracle.mm_i4(a, q, s.astype(np.float32), k, g))
    same(ctx.upload_q4a(q, s, mn, k, g).mm(a), oracle.mm_q4a(a, q, s.astype(np.float32), mn.astype(np.float32), k, g))


def test_non_finite_and_subnormal_values(ctx):
    rng = np.random.default_rng(5)
    m, k, n, g = 20, 300, 40, 32
    a = rng.standard_normal((m, k), dtype=np.float32)
    a[0, 299], a[1, 7], a[2, 255], a[3] = np.inf, -np.inf, 3e38, a[3] * np.float32(1e-38)
    a[4, 3], a[5] = np.nan, 0.0
    a[6, 256:] = -0.0
    q, s, mn = packed_weight(rng, n, k, g)
    got, ref = ctx.upload_i4(q, s, k, g).mm_exact(a), oracle.mm_i4(a, q, s.astype(np.float32), k, g)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    fin = ~np.isnan(ref)
    same(got[fin], ref[fin])


@pytest.mark.parametrize("g,k", [(32, 40), (64, 200), (48, 104), (32, 320)])
@pytest.mark.parametrize("m,n", [(2, 16), (33, 70)])
def test_non_finite_scales(ctx, m, n, k, g):
    """A group scale that is infinite or NaN: s4 * scale in each weight, so a
    group whose products share a sign sums to that infinity (the short last
    group of rows of one nibble, whose activations are positive), a zero
    nibble or both signs to NaN."""
    rng = np.random.default_rng(m + n + k + g)
    a = rng.uniform(0.5, 1.5, (m, k)).astype(np.float32)
    q, s, mn = packed_weight(rng, n, k, g)
    last = (k - 1) // g
    for row, (scale, byte) in enumerate([(np.inf, 0x33), (np.inf, 0xDD), (-np.inf, 0x33), (-np.inf, 0x88), (np.inf, 0x30),
                                         (np.nan, 0x33), (np.inf, 0x3D), (-np.inf, 0x7F)]):
        q[row, last * g // 2:] = byte
        s[row, last] = scale
    s[8, 0], s[9, 0] = np.inf, np.nan  # a whole group of mixed nibbles
    f32 = lambda v: v.astype(np.float32)
    with np.errstate(invalid="ignore"):
        for got, ref in ((ctx.upload_i4(q, s, k, g).mm_exact(a), oracle.mm_i4(a, q, f32(s), k, g)),
                         (ctx.upload_q4a(q, s, mn, k, g).mm(a), oracle.mm_q4a(a, q, f32(s), f32(mn), k, g))):
            assert np.isinf(ref[:, :4]).all() and np.isnan(ref[:, 5]).all()
            assert np.array_equal(np.isnan(got), np.isnan(ref))
            same(got[~np.isnan(ref)], ref[~np.isnan(ref)])


@pytest.mark.parametrize("dtype", ["f16", "f32", "q4a", "i4"])
@pytest.mark.parametrize("T,topk,d,mi", [(1, 2, 288, 70), (4, 2, 96, 33), (5, 3, 256, 17), (90, 2, 520, 64),
                                         (200, 1, 64, 300)])
def test_expert_banks_in_a_dot_order(ctx, dtype, T, topk, d, mi):
    E, rng = 4, np.random.default_rng(T + d + mi)
    g = 20 if dtype == "i4" else 32  # an i4 group with no digit form

    def mat(i, o):
        if dtype in ("f16", "f32"):
            w = (rng.standard_normal((i, o), dtype=np.float32) * np.float32(0.05))
            return {"raw": w.astype(np.float16).view(np.uint16) if dtype == "f16" else w, "scale": None, "min": None}
        q, s, mn = packed_weight(rng, o, i, g)
        return {"raw": q, "scale": s.view(np.uint16), "min": mn.view(np.uint16) if dtype == "q4a" else None}

    gate, up, down = ([mat(i, o) for _ in range(E)] for i, o in ((d, mi), (d, mi), (mi, d)))
    col = lambda ms, key: None if ms[0][key] is None else [m[key] for m in ms]
    bank = ctx.upload_moe(dtype, d, mi, col(gate, "raw"), col(down, "raw"), col(up, "raw"), col(gate, "scale"),
                          col(up, "scale"), col(down, "scale"), col(gate, "min"), col(up, "min"), col(down, "min"),
                          g=0 if dtype in ("f16", "f32") else g)
    x = rng.standard_normal((T, d), dtype=np.float32)
    for which, ms, (i, o) in ((0, gate, (d, mi)), (2, down, (mi, d))):
        xi = rng.standard_normal((T, i), dtype=np.float32)
        f = lambda v: None if v is None else v.view(np.float16).astype(np.float32)
        w = oracle.expert(dtype, ms[1]["raw"], f(ms[1]["scale"]), f(ms[1]["min"]), g, i, o)
        same(bank.expert_mm(which, 1, xi), oracle.expert_mm(xi, w))
    lg = rng.standard_normal((T, E)).astype(np.float32)
    per_row = np.stack([bank.forward(x[t:t + 1], lg[t:t + 1], topk)[0] for t in range(T)])
    same(bank.forward(x, lg, topk), per_row)  # tiles of 4 and of 32 rows, one expert's rows alone or together


@pytest.mark.parametrize("g", [32, 64, 13, 1, 4000])
@pytest.mark.parametrize("k,n", [(1, 3), (31, 5), (33, 300), (255, 64), (790, 1), (1001, 700), (6346, 184), (2304, 129),
                                 (16383, 17), (16400, 9), (64, 70), (65, 70), (895, 40), (897, 40), (790, 4096),
                                 (8191, 20), (8193, 20)])
def test_one_row_of_any_width_and_group(ctx, k, n, g):
    """M == 1 where the aligned kernels do not apply: the AVX2 orders, groups
    that start inside a byte, rows too long for LDS."""
    rng = np.random.default_rng(k + n + g)
    a = rng.standard_normal((1, k), dtype=np.float32)
    q, s, mn = packed_weight(rng, n, k, g)
    same(ctx.upload_i4(q, s, k, g).mm_exact(a), oracle.mm_i4(a, q, s.astype(np.float32), k, g))
    if (k + g - 1) // g <= 8192:  # q4a: one row's group terms must fit in LDS
        same(ctx.upload_q4a(q, s, mn, k, g).mm(a),
             oracle.mm_q4a(a, q, s.astype(np.float32), mn.astype(np.float32), k, g))
