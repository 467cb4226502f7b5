"""GPU parity of lgmlh_flash_attn (graph:flash_attn over strided K / V
views with an explicit mask) against the oracle's orc_flash_attn (pinned in
tests/test_oracle_flash.py), within 1e-5 max relative error (the bar is
2e-3): head sizes 16..256, GQA, random and causal masks with broadcast
planes, softcap, ALiBi, a fully masked row, pool-row views with strides.
Under the fill_blocks mask over the pool rows it equals the paged kernel
(lgmlh_paged_attention) on the same cells.
"""
import ctypes as C

import numpy as np
import pytest

from oracle import core, kvpool as kp
from tests.gpu_util import rel_err

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def L():
    from lgml_amd import hip
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return hip.lib()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def st():
    return torch.cuda.current_stream().cuda_stream


def gpu_flash(L, q, k, v, Hkv, n_kv, k_strides, v_strides, mask, scale, max_bias=0.0,
              softcap=0.0):
    from lgml_amd import hip
    H, T, D = q.shape
    qd, kd, vd = dev(q), dev(k), dev(v)
    md = dev(mask) if mask is not None else None
    mh, mr = (mask.shape[0], mask.shape[1]) if mask is not None else (0, 0)
    out = torch.full((T, H, D), float("nan"), dtype=torch.float32, device="cuda")
    hip.check(L.lgmlh_flash_attn(qd.data_ptr(), H, T, D, kd.data_ptr(), vd.data_ptr(), Hkv, n_kv,
                                 k_strides[0], k_strides[1], v_strides[0], v_strides[1],
                                 md.data_ptr() if md is not None else None, mh, mr, scale,
                                 max_bias, softcap, out.data_ptr(), st()))
    return out.cpu().numpy()


CASES = [  # H, Hkv, T, D, n_kv, mask kind, softcap, max_bias
    (4, 2, 5, 16, 37, "random", 0.0, 0.0),
    (8, 8, 3, 32, 200, "causal", 0.0, 0.0),
    (8, 2, 17, 64, 129, "random", 20.0, 0.0),
    (12, 4, 4, 80, 70, "random", 0.0, 8.0),
    (32, 8, 9, 128, 300, "causal", 0.0, 0.0),
    (8, 4, 2, 256, 1100, "random", 0.0, 0.0),
    (4, 1, 6, 128, 65, None, 0.0, 0.0),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_flash_attn_matches_oracle(L, case):
    H, Hkv, T, D, n_kv, kind, softcap, max_bias = CASES[case]
    rng = np.random.default_rng(10 + case)
    q = (rng.standard_normal((H, T, D)) * 0.5).astype(np.float32)
    k = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    v = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    mask = None
    if kind == "random":
        planes = 2 if H % 2 == 0 else 1
        m = rng.standard_normal((planes, T + 1, n_kv)).astype(np.float32)
        m[rng.random(m.shape) < 0.4] = -np.inf
        m[-1, T - 1, :] = -np.inf  # a fully masked row
        mask = core.f32_to_f16_bits(m)
    elif kind == "causal":
        m = np.where(np.arange(n_kv)[None, :] <= n_kv - T + np.arange(T)[:, None], 0.0, -np.inf)
        mask = core.f32_to_f16_bits(m[None].astype(np.float32))
    scale = 1.0 / np.sqrt(D)
    print("flash_attn case %d: H=%d Hkv=%d T=%d D=%d n_kv=%d mask=%s softcap=%g max_bias=%g" % (
        case, H, Hkv, T, D, n_kv, kind, softcap, max_bias), flush=True)
    got = gpu_flash(L, q, k, v, Hkv, n_kv, (D, n_kv * D), (D, n_kv * D), mask, scale, max_bias,
                    softcap)
    want = core.flash_attn(q, k, v, Hkv, mask, scale, max_bias, softcap)
    assert np.isfinite(got).all()
    assert rel_err(got.reshape(T * H, D) + 1e-30, want.reshape(T * H, D) + 1e-30) < 1e-5
    if kind == "random":
        assert not got[T - 1, H - 1].any()  # the fully masked row is zeros


def test_flash_attn_on_pool_rows_equals_paged_attention(L):
    """The same cells as plain (cap, Hkv * D) rows under fill_blocks masks
    and as the block pool through the plan give the same outputs."""
    from lgml_amd import hip, runtime
    rng = np.random.default_rng(3)
    H, Hkv, D, B, cap = 32, 8, 128, 64, 2048
    pool = kp.Pool(cap // B, B)
    seqs = [kp.Seq(pool) for _ in range(3)]
    seq_n, npast = [1, 9, 1], [700, 100, 5]
    for s in seqs:
        kp.reserve(s, 65)
    for s, n, p in zip(seqs, seq_n, npast):
        kp.reserve(s, n + p)
    bt = np.full((3, max(len(s.blocks) for s in seqs)), -1, np.int32)
    for i, s in enumerate(seqs):
        bt[i, :len(s.blocks)] = s.blocks
    krows = core.f32_to_f16_bits(rng.standard_normal((cap, Hkv * D)).astype(np.float32))
    vrows = core.f32_to_f16_bits(rng.standard_normal((cap, Hkv * D)).astype(np.float32))
    N = sum(seq_n)
    q = rng.standard_normal((N, H, D)).astype(np.float32)
    # the paged kernel on the block pool
    plan = runtime.Plan(seq_n, npast, bt, np.zeros(N, np.int32), H, Hkv, cap // B)
    kb = L.lgmlh_kv_layer_bytes(cap, Hkv, D)
    kpd = torch.zeros(kb, dtype=torch.uint8, device="cuda")
    vpd = torch.zeros(kb, dtype=torch.uint8, device="cuda")
    allc = np.arange(cap, dtype=np.int64)
    kf, vf, cd = dev(core.f16_bits_to_f32(krows)), dev(core.f16_bits_to_f32(vrows)), dev(allc)
    hip.check(L.lgmlh_kv_store(kpd.data_ptr(), vpd.data_ptr(), cap, Hkv, D, kf.data_ptr(),
                               vf.data_ptr(), cd.data_ptr(), allc.ctypes.data, cap, st()))
    paged = torch.empty((N, H, D), dtype=torch.float32, device="cuda")
    wsb = L.lgmlh_attention_workspace(C.byref(plan.info), D)
    ws = torch.empty(max(wsb, 1), dtype=torch.uint8, device="cuda")
    qd = dev(q)
    hip.check(L.lgmlh_paged_attention(qd.data_ptr(), H, Hkv, D, 1.0 / np.sqrt(D), kpd.data_ptr(),
                                      vpd.data_ptr(), C.byref(plan.ub), paged.data_ptr(),
                                      ws.data_ptr(), wsb, st()))
    paged = paged.cpu().numpy()
    off = 0
    for i, (n, p) in enumerate(zip(seq_n, npast)):
        m16 = core.f32_to_f16_bits(kp.fill_blocks(n, cap, p, B, list(seqs[i].blocks)))[None]
        qh = np.ascontiguousarray(q[off:off + n].transpose(1, 0, 2))
        got = gpu_flash(L, qh, krows, vrows, Hkv, cap, (Hkv * D, D), (Hkv * D, D), m16,
                        1.0 / np.sqrt(D))
        assert rel_err(got.reshape(n * H, D), paged[off:off + n].reshape(n * H, D)) < 1e-5, i
        off += n


# Edges of the kernel's tiles: cells around 32 and 64 and the groups that
# share them, rows around 16 and 64 (the last two cases: from 96 workgroups
# of 64 rows, four row tiles each), head sizes that are and are not whole
# MFMA steps. The bound is the one of the other cases: hi + lo pairs carry 22
# bits of these scores and probabilities, so products and their f32 sums over
# up to 256 + 300 terms stay within 556 * 2^-24 + 2^-21 of the largest term,
# 3.4e-5; errors add at random and measure 4e-7.
EDGES = [  # H, Hkv, T, D, n_kv
    (1, 1, 1, 8, 1), (3, 1, 5, 16, 31), (2, 2, 16, 40, 32), (4, 1, 4, 64, 33), (4, 2, 9, 96, 63),
    (2, 1, 8, 128, 64), (8, 2, 1, 128, 65), (2, 1, 3, 160, 129), (2, 2, 17, 192, 255),
    (8, 1, 2, 256, 257), (32, 32, 129, 72, 130), (16, 8, 395, 128, 70), (8, 8, 800, 256, 40),
]


@pytest.mark.parametrize("case", range(len(EDGES)))
def test_flash_attn_tile_edges(L, case):
    H, Hkv, T, D, n_kv = EDGES[case]
    rng = np.random.default_rng(50 + case)
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    v = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    m = np.where(rng.random((1, T, n_kv)) < 0.5, 0.0, -np.inf).astype(np.float32)
    m[0, :, 0] = 0.5
    mask = core.f32_to_f16_bits(m)
    print("flash_attn edge %d: H=%d Hkv=%d T=%d D=%d n_kv=%d" % (case, H, Hkv, T, D, n_kv),
          flush=True)
    got = gpu_flash(L, q, k, v, Hkv, n_kv, (D, n_kv * D), (D, n_kv * D), mask, D ** -0.5)
    want = core.flash_attn(q, k, v, Hkv, mask, D ** -0.5, 0.0, 0.0)
    assert rel_err(got.reshape(T * H, D), want.reshape(T * H, D)) < 1e-5


@pytest.mark.parametrize("T", [3, 500])
def test_flash_attn_masked_cells_hold_anything(L, T):
    """Cells that a row does not see may hold infinities and NaN in K and V;
    a V value that is not finite reaches exactly the rows that see its cell;
    rows whose every mask value is f16's lowest; f32 rows of q beyond f16."""
    rng = np.random.default_rng(60)
    H, Hkv, D, n_kv = 16, 8, 64, 150
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    q[1] *= 3e5
    k = rng.standard_normal((Hkv, n_kv, D)).astype(np.float32)
    k[2:4] *= 1e-5  # heads 4..7: scores in range at q scaled up
    v = rng.standard_normal((Hkv, n_kv, D)).astype(np.float32)
    m = np.where(rng.random((1, T, n_kv)) < 0.3, -np.inf, 0.0).astype(np.float32)
    m[0, :, 100:] = -np.inf
    m[0, 0, :100] = -65504.0
    m[0, :, 5] = 0.0
    m[0, 1, 5] = -np.inf
    clean = core.flash_attn(q, core.f32_to_f16_bits(k), core.f32_to_f16_bits(v), Hkv,
                            core.f32_to_f16_bits(m), 0.125, 0.0, 0.0)
    k[:, 100:], v[:, 100:] = np.nan, np.inf
    v[:, 120] = np.nan
    v[0, 5, 7] = np.inf  # heads 0 and 1, every row but row 1
    got = gpu_flash(L, q, core.f32_to_f16_bits(k), core.f32_to_f16_bits(v), Hkv, n_kv,
                    (D, n_kv * D), (D, n_kv * D), core.f32_to_f16_bits(m), 0.125)
    sees = np.ones((T, H), bool)
    sees[1] = False
    sees[:, 2:] = False
    # rows of head 1 put all weight on one cell: whether p of cell 5 is
    # above 0 is theirs, so only head 0 is asserted to hold the infinity
    assert np.isinf(got[sees[:, 0], 0, 7]).all() and np.isfinite(got[1]).all()
    got[:, :2, 7], clean[:, :2, 7] = 0, 0
    assert rel_err(got.reshape(T * H, D), clean.reshape(T * H, D)) < 1e-5


def softmax64(s, v):
    """Rows of softmax(s) v in f64 (s (rows, cells), v (cells, D))."""
    p = np.exp(s - s.max(axis=1, keepdims=True))
    return p @ v.astype(np.float64) / p.sum(axis=1, keepdims=True)


# One cell that takes almost all of a row's weight, above thousands of others
# whose sum is the result (the cell's V is 0) or a part of it. Scores are
# exact (one value of q and k), so a row loses: its argument of exp2, |s|
# log2(e) <= 26, rounded to f32 (2^-20 ln 2 = 6.6e-7) with log2(e) itself
# (2e-7), P's 22 bits and exp2's last bit (2.4e-7 each), and a rounding of l and
# O per turn (16 rows: 8 groups of 32 cells; 1024 rows: 2 groups of 64). The
# sums are alike from row to row, so the roundings may all go one way. It
# measures a third to a half of the bound.
@pytest.mark.parametrize("n_kv", [2048, 32768])
@pytest.mark.parametrize("T", [16, 1024])
@pytest.mark.parametrize("sink_v", [0, 1])
def test_flash_attn_one_cell_above_thousands(L, n_kv, T, sink_v):
    rng = np.random.default_rng(63)
    H, Hkv, D = 8, 8, 32
    gaps = np.linspace(1, 16, T).astype(np.float16).astype(np.float32)  # a gap per row
    q = np.zeros((H, T, D), np.float32)
    q[:, :, 3] = gaps
    k = np.zeros((n_kv, Hkv, D), np.float16)
    k[5, :, 3] = 1.0
    k[7::7, :, 3] = -0.125
    v = rng.standard_normal((n_kv, Hkv, D)).astype(np.float16)
    v[5] *= sink_v
    got = gpu_flash(L, q, k.view(np.uint16), v.view(np.uint16), Hkv, n_kv, (Hkv * D, D),
                    (Hkv * D, D), None, 1.0)
    for h in range(H):
        want = softmax64(gaps[:, None].astype(np.float64) * k[None, :, h, 3].astype(np.float64),
                         v[:, h])
        err = np.linalg.norm(got[:, h] - want, axis=1) / np.linalg.norm(want, axis=1)
        turns = n_kv // (32 * 8 if T == 16 else 64 * 2)
        assert err.max() < 1.4e-6 + turns * 2.0 ** -23, (h, gaps[err.argmax()], err.max())


@pytest.mark.parametrize("T", [3, 500])
@pytest.mark.parametrize("size", [1.0, 1e-36, 1e30])
def test_flash_attn_one_value_of_q_far_above_the_others(L, T, size):
    """Rows of q whose largest value meets zeros in K: the others, 2^-14 to
    2^-22 of it, make the scores, and pairs hold 22 bits of them. With D = 64
    products and sums of up to 200 terms the bound is that of the tile edges;
    rows far from 1 in size are scaled the same way."""
    rng = np.random.default_rng(64)
    H, Hkv, D, n_kv = 16, 8, 64, 200
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    q[:, :, 3] = 2.0 ** rng.integers(14, 23, (H, T))
    k = rng.standard_normal((n_kv, Hkv, D)).astype(np.float16)
    k[:, :, 3] = 0
    v = rng.standard_normal((n_kv, Hkv, D)).astype(np.float16)
    q = (q * np.float32(size)).astype(np.float32)
    scale = float(np.float32(0.125 / size))
    got = gpu_flash(L, q, k.view(np.uint16), v.view(np.uint16), Hkv, n_kv, (Hkv * D, D),
                    (Hkv * D, D), None, scale)
    for h in range(H):
        s = q[h].astype(np.float64) @ k[:, h // 2].astype(np.float64).T * scale
        assert rel_err(got[:, h], softmax64(s, v[:, h // 2])) < 1e-5, h


@pytest.mark.parametrize("softcap", [0.0, 20.0])
@pytest.mark.parametrize("T,D", [(3, 64), (500, 64), (4, 128), (400, 128), (3, 256)])
def test_flash_attn_seen_infinities_in_q_and_k(L, T, D, softcap):
    """A score of -inf drops its cell, one of +inf or NaN makes its row NaN;
    with a softcap infinite scores are +- softcap. K holds infinities that
    rows see (q with and without a low part, or 0, beside them), and so does q."""
    rng = np.random.default_rng(65)
    H, Hkv, n_kv = 16, 8, 150
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    q[:, :, 3:5] = np.abs(q[:, :, 3:5])
    q[3::4] = q[3::4].astype(np.float16)
    q[2, :, 3] *= -1        # +inf at cell 5
    q[4, 0, 4] = 0          # 0 * inf at cell 77
    q[5, 1, 7] = np.inf     # K is below 0 there: no cell left
    q[7, 2, 8] = -np.inf    # and of both signs here
    k = rng.standard_normal((n_kv, Hkv, D)).astype(np.float16)
    k[:, :, 7] = -np.abs(k[:, :, 7])
    k[5, :, 3] = -np.inf
    k[77, :, 4] = -np.inf
    k[130, 6] = np.nan
    v = rng.standard_normal((n_kv, Hkv, D)).astype(np.float16)
    got = gpu_flash(L, q, k.view(np.uint16), v.view(np.uint16), Hkv, n_kv, (Hkv * D, D),
                    (Hkv * D, D), None, D ** -0.5, 0.0, softcap)
    n_nan = 0
    with np.errstate(invalid="ignore"):
        for h in range(H):
            s = (q[h].astype(np.float64)[:, None] * k[None, :, h // 2].astype(np.float64)).sum(2)
            s = s * D ** -0.5
            s = softcap * np.tanh(s / softcap) if softcap else s
            want = softmax64(s, v[:, h // 2])
            want[s.max(axis=1) == -np.inf] = 0  # no cell left
            bad = np.isnan(want).any(axis=1)
            assert np.isnan(got[bad, h]).all() and np.isfinite(got[~bad, h]).all(), h
            assert not (~bad).any() or rel_err(got[~bad, h], want[~bad]) < 1e-5, h
            n_nan += int(bad.sum())
    assert 2 * T < n_nan < 4 * T  # heads 12 and 13, which see the NaN, and single rows


# The switch between a wave per row and tiles: up to 4 cells of 2048 rows in all,
# for heads past 32 up to 8 cells of 512 rows.
@pytest.mark.parametrize("H,Hkv,T,D,n_kv", [
    (4, 2, 512, 16, 1), (4, 2, 513, 16, 2), (4, 1, 512, 40, 4), (4, 2, 3, 40, 5),
    (8, 2, 64, 64, 5), (8, 2, 65, 64, 8), (2, 1, 256, 128, 8), (2, 1, 5, 128, 9),
    (8, 8, 1, 256, 3), (6, 2, 11, 200, 7)])
def test_flash_attn_few_cells(L, H, Hkv, T, D, n_kv):
    rng = np.random.default_rng(66)
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    v = rng.standard_normal((Hkv, n_kv, D)).astype(np.float32)
    m = np.where(rng.random((2, T, n_kv)) < 0.5, rng.random((2, T, n_kv)), -np.inf)
    m[:, :, 0] = 0.25
    m[1, T - 1] = -np.inf  # a row that sees nothing
    mask = core.f32_to_f16_bits(m.astype(np.float32))
    want = core.flash_attn(q, k, core.f32_to_f16_bits(v), Hkv, mask, D ** -0.5, 2.0, 15.0)
    if n_kv > 1:  # what no row sees may hold anything
        m[:, :, n_kv - 1] = -np.inf
        mask = core.f32_to_f16_bits(m.astype(np.float32))
        want = core.flash_attn(q, k, core.f32_to_f16_bits(v), Hkv, mask, D ** -0.5, 2.0, 15.0)
        v[:, n_kv - 1] = np.nan
    got = gpu_flash(L, q, k, core.f32_to_f16_bits(v), Hkv, n_kv, (D, n_kv * D), (D, n_kv * D), mask,
                    D ** -0.5, 2.0, 15.0)
    assert rel_err(got.reshape(T * H, D) + 1e-30, want.reshape(T * H, D) + 1e-30) < 1e-5


@pytest.mark.parametrize("H,Hkv,T,D,n_kv,parts", [
    (32, 8, 200, 64, 300, (1, 176, 177)),  # 4 row tiles of 16 a workgroup from 177 rows up
    (8, 8, 300, 128, 6, (64, 65, 300))])   # a wave per row up to 64 rows
def test_flash_attn_rows_in_calls_of_other_sizes(L, H, Hkv, T, D, n_kv, parts):
    """A row's last bits depend on the kernel that the number of rows picks:
    within the f32 bound of the tile edges it is the same in any call."""
    rng = np.random.default_rng(67)
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    v = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    whole = gpu_flash(L, q, k, v, Hkv, n_kv, (D, n_kv * D), (D, n_kv * D), None, D ** -0.5)
    for n in parts:
        some = gpu_flash(L, np.ascontiguousarray(q[:, :n]), k, v, Hkv, n_kv, (D, n_kv * D),
                         (D, n_kv * D), None, D ** -0.5)
        assert rel_err(some.reshape(n * H, D), whole[:n].reshape(n * H, D)) < 1e-5, n


def test_flash_attn_addresses_of_elements(L):
    """q, v, the mask and out start at any element (k is 16-byte aligned)."""
    from lgml_amd import hip
    rng = np.random.default_rng(61)
    H, Hkv, T, D, n_kv = 4, 2, 20, 48, 77
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    k = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    v = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D + 1)).astype(np.float32))
    m = core.f32_to_f16_bits(np.where(rng.random((1, T, n_kv)) < 0.5, 0, -1).astype(np.float32))
    qd, kd = dev(np.concatenate([np.zeros(1, np.float32), q.ravel()])), dev(k)
    vd = dev(np.concatenate([np.zeros(1, np.uint16), v.ravel()]).view(np.int16))
    md = dev(np.concatenate([np.zeros(3, np.uint16), m.ravel()]).view(np.int16))
    out = torch.zeros(T * H * D + 1, dtype=torch.float32, device="cuda")
    hip.check(L.lgmlh_flash_attn(qd.data_ptr() + 4, H, T, D, kd.data_ptr(), vd.data_ptr() + 2, Hkv,
                                 n_kv, D, n_kv * D, D + 1, n_kv * (D + 1), md.data_ptr() + 6, 1, T,
                                 0.2, 0.0, 0.0, out.data_ptr() + 4, st()))
    want = core.flash_attn(q, k, np.ascontiguousarray(v[:, :, :D]), Hkv, m, 0.2, 0.0, 0.0)
    got = out.cpu().numpy()
    assert got[0] == 0
    assert rel_err(got[1:].reshape(T * H, D), want.reshape(T * H, D)) < 1e-5


def test_flash_attn_rows_near_the_largest_f32(L):
    """q of up to 3.4e38 (past the exponents a power of two brings to 1)."""
    rng = np.random.default_rng(62)
    H, Hkv, T, D, n_kv = 2, 1, 5, 16, 40
    q = rng.standard_normal((H, T, D)).astype(np.float32)
    q[0] = np.sign(q[0]) * rng.uniform(0.5, 1.0, (T, D)).astype(np.float32) * np.float32(3.4e38)
    k = core.f32_to_f16_bits(1e-3 * rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    v = core.f32_to_f16_bits(rng.standard_normal((Hkv, n_kv, D)).astype(np.float32))
    m = core.f32_to_f16_bits(np.zeros((1, T, n_kv), np.float32))
    got = gpu_flash(L, q, k, v, Hkv, n_kv, (D, n_kv * D), (D, n_kv * D), m, 0.25)
    want = core.flash_attn(q, k, v, Hkv, m, 0.25, 0.0, 0.0)
    assert rel_err(got.reshape(T * H, D), want.reshape(T * H, D)) < 1e-5


def test_flash_attn_more_row_tiles_than_a_grid_has_in_y(L):
    """65537 workgroups of 64 rows: the last ones write their rows too."""
    from lgml_amd import hip
    H, D = 8, 8
    T = 65536 * 8 + 3
    q = torch.ones(H * T * D, device="cuda")
    k = torch.ones(D, dtype=torch.float16, device="cuda")
    v = torch.arange(D, dtype=torch.float16, device="cuda")
    out = torch.full((T * H, D), -1.0, device="cuda")
    hip.check(L.lgmlh_flash_attn(q.data_ptr(), H, T, D, k.data_ptr(), v.data_ptr(), 1, 1, D, D, D,
                                 D, 0, 1, T, 0.5, 0.0, 0.0, out.data_ptr(), st()))
    assert bool((out == torch.arange(D, device="cuda").float()).all())


def test_flash_attn_more_rows_than_an_int_counts(L):
    """2^31 + 192 (token, query head) pairs of one KV head."""
    from lgml_amd import hip
    H, D, T = 64, 8, 2 ** 25 + 3
    if torch.cuda.mem_get_info()[0] < 2 * H * T * D * 4 + (8 << 30):
        pytest.skip("needs 137 GB")
    q = torch.ones(H * T * D, device="cuda")
    k = torch.ones(D, dtype=torch.float16, device="cuda")
    v = torch.arange(1, D + 1, dtype=torch.float16, device="cuda")
    out = torch.zeros(T * H, D, device="cuda")
    hip.check(L.lgmlh_flash_attn(q.data_ptr(), H, T, D, k.data_ptr(), v.data_ptr(), 1, 1, D, D, D,
                                 D, 0, 1, T, 0.5, 0.0, 0.0, out.data_ptr(), st()))
    want = torch.arange(1, D + 1, device="cuda").float()
    for at in (0, 2 ** 30, 2 ** 31 - 4096, T * H - 4096):
        assert bool((out[at:at + 4096] == want).all()), at
    del q, out
    torch.cuda.empty_cache()
