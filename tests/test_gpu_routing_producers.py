"""GPU parity: device-side MoE routing / packing (src/ops/moe.cpp:22-216,366-446,
src/model/qwen3moe_pack.cpp) and the fused normalisation -> block_q8_1x producers
(src/ops/elementwise.cpp:136-191, src/ops/deltanet.cpp:73-130)."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import check, dev, host

pytestmark = pytest.mark.gpu


def f16(a):
    return O.round_fp16(np.asarray(a, np.float32))


@pytest.mark.parametrize("T,E,k,H", [(1, 256, 8, 2048), (5, 128, 8, 512), (33, 32, 4, 2880), (2, 1000, 64, 256)])
def test_moe_router(mx, T, E, k, H):
    x = f16(O.normal(9100, (T, H)))
    Wg = O.normal(9101, (E, H), 0.0, 0.05).astype(np.float32)
    idx, w = mx.ops.moe_router(dev(x).half(), dev(Wg), E, k)
    logits = (x.astype(np.float64) @ Wg.astype(np.float64).T).astype(np.float32)
    ids_ref, w_ref = O.route_from_logits(logits, k)
    idx_h, w_h = host(idx), host(w).astype(np.float32)
    # a pick may differ only where two probabilities tie within fp32 noise of the logits
    same = (idx_h == ids_ref).all(axis=1)
    assert same.mean() >= 0.9, "routing disagrees on %d of %d tokens" % ((~same).sum(), T)
    assert (np.diff(idx_h, axis=1) > 0).all(), "expert ids ascending and distinct"
    np.testing.assert_allclose(w_h.sum(axis=1), 1.0, atol=4e-3)
    check(w_h[same], w_ref[same], "router weights", max_rel=2e-3)


@pytest.mark.parametrize("T,E,k", [(1, 32, 4), (7, 128, 8), (3, 1024, 16)])
def test_moe_topk_from_logits(mx, T, E, k):
    logits = f16(O.normal(9200, (T, E), 0.0, 2.0))
    idx, w = mx.ops.moe_topk_from_logits(dev(logits).half(), k)
    ids_ref, w_ref = O.route_from_logits(logits, k)
    idx_h = host(idx)
    same = (idx_h == ids_ref).all(axis=1)
    # fp16 logits tie exactly now and then; the reference breaks an exact tie towards the higher id
    for t in np.where(~same)[0]:
        a, b = set(idx_h[t]) - set(ids_ref[t]), set(ids_ref[t]) - set(idx_h[t])
        assert len(a) == len(b) and sorted(logits[t, list(a)]) == sorted(logits[t, list(b)]), "differs beyond an exact tie"
    check(host(w).astype(np.float32)[same], w_ref[same], "topk weights", max_rel=2e-3)


def test_moe_topk_tie_goes_to_higher_id(mx):
    logits = np.zeros((1, 64), np.float32)
    logits[0, [3, 9, 20, 41]] = 1.0          # four-way exact tie, k = 2 -> ids 20 and 41
    idx, w = mx.ops.moe_topk_from_logits(dev(logits).half(), 2)
    assert host(idx).tolist() == [[20, 41]]
    np.testing.assert_allclose(host(w).astype(np.float32), [[0.5, 0.5]], atol=1e-3)


def test_moe_router_nan_payload_keeps_ids_in_range(mx):
    """Every bit of a NaN set (the largest key there is): each token still gets k distinct ids of the bank."""
    Wg = torch.full((8, 256), -1, dtype=torch.int32).view(torch.float32)
    idx, _ = mx.ops.moe_router(dev(np.ones((2, 256), np.float32)).half(), Wg.cuda(), 8, 4)
    assert host(idx).tolist() == [[4, 5, 6, 7]] * 2


def test_moe_topk_weights_are_rounded_twice(mx):
    """p * (1 / sum) is an fp32 value before it is an fp16 one: tokens whose fp32 product lies on the midpoint of
    two halves while the unrounded product does not, so that one rounding would give the other half.  Bits pinned from the kernel that
    kept the weights in fp32 in LDS."""
    rows = [(0xB92C, 0x3B64, 0xB834, 0xBC45, 0x40A1, 0x377F), (0x3C55, 0xC098, 0x3FC0, 0xC2F2, 0x34D8, 0xC4B5), (0x411D, 0xBD95, 0x3773, 0x31CB, 0xC097, 0xC17E),
            (0xA993, 0xBCF1, 0x3FF5, 0xC16A, 0xB558, 0xB86D), (0xBB45, 0x30CA, 0xC2C2, 0x3D73, 0xBE2E, 0xBBCA), (0x3D46, 0xC0CA, 0xBACC, 0x3E00, 0xB9FC, 0x4037)]
    ids = [(1, 4, 5), (0, 2, 4), (0, 2, 3), (0, 2, 4), (0, 1, 3), (0, 3, 5)]
    bits = [(0x31AA, 0x39B0, 0x2F2F), (0x3434, 0x38F0, 0x2FB4), (0x3A94, 0x2E80, 0x2CE4), (0x2ED2, 0x3A82, 0x2D1A), (0x2CB7, 0x32CC, 0x39B6), (0x3346, 0x345C, 0x3800)]
    idx, w = mx.ops.moe_topk_from_logits(dev(np.array(rows, np.uint16).view(np.float16)), 3)
    assert host(idx).tolist() == [list(r) for r in ids]
    assert host(w).view(np.uint16).tolist() == [list(r) for r in bits]


@pytest.mark.parametrize("T,E,K", [(1, 32, 4), (64, 8, 2), (300, 128, 8), (2048, 128, 8)])
def test_moe_packing_device_equals_host(mx, T, E, K):
    rng = np.random.default_rng(T + E)
    p = np.arange(1, E + 1, dtype=np.float64) ** -1.1
    p /= p.sum()
    ids = np.stack([np.sort(rng.choice(E, size=K, replace=False, p=p)) for _ in range(T)]).astype(np.int32)
    w = f16(rng.random((T, K)).astype(np.float32))
    off_r, si_r, wp_r, t2p_r = O.build_moe_packing(ids, w, E)
    for decode in ([False, True] if T == 1 else [False]):
        off, si, wp, t2p = mx.ops.moe_build_packing_device(dev(ids), dev(w).half(), E, decode=decode)
        assert np.array_equal(host(off).view(np.uint32), off_r)
        assert np.array_equal(host(si), si_r)
        assert np.array_equal(host(t2p), t2p_r)
        assert np.array_equal(host(wp).astype(np.float32), wp_r)


def _fma32(a, b, c):
    """fp32 fused multiply-add of fp32 a, c and fp16-valued b: the product is exact in 64 bits, the sum is rounded to odd there (so
    that rounding it again to fp32 is one correct rounding)."""
    p, c = a.astype(np.float64) * b, c.astype(np.float64)
    s = p + c
    t = s - p
    err = (p - (s - t)) + (c - t)
    odd = (s.view(np.int64) & 1) == 1
    s = np.where((err != 0) & ~odd, np.nextafter(s, np.where(err > 0, np.inf, -np.inf)), s)
    return s.astype(np.float32)


def router_logits(x, W):
    """The documented order of the router's sums: lane l takes elements 4 l .. 4 l + 3 of every 256, then a tree of neighbours."""
    T, H = x.shape
    acc = np.zeros((T, len(W), 64), np.float32)
    for c in range(0, H, 256):
        n = min(256, H - c) // 4
        xs, ws = x[:, None, c:c + 4 * n].reshape(T, 1, n, 4), W[None, :, c:c + 4 * n].reshape(1, len(W), n, 4)
        d = (ws[..., 1].astype(np.float64) * xs[..., 1]).astype(np.float32)
        for i in (0, 2, 3):
            d = _fma32(np.broadcast_to(ws[..., i], d.shape), xs[..., i], d)
        acc[..., :n] += d
    while acc.shape[-1] > 1:
        acc = acc[..., 0::2] + acc[..., 1::2]
    return acc[..., 0]


@pytest.mark.parametrize("T,E,H", [(1, 33, 2880), (3, 32, 36), (60, 65, 264), (64, 128, 1028), (333, 60, 516), (65, 128, 256), (1030, 65, 260), (64, 1024, 256)])
def test_moe_router_logits_do_not_depend_on_the_call(mx, T, E, H):
    """Every tile size of the logits kernel (1 x 1, 2 x 2, 4 x 4, 8 x 8 by T * E), whole and partial pieces, ragged tiles: the bits of
    the one summation order, also for a token alone and for rows on an 8-byte boundary."""
    x = f16(O.normal(9170 + T, (T, H)))
    Wg = O.normal(9171 + E, (E, H), 0.0, 1.0 / np.sqrt(H)).astype(np.float32)
    flat = torch.zeros(T * H + 4, dtype=torch.float16, device="cuda")
    flat[4:] = dev(x).half().reshape(-1)
    k = min(4, E)

    def logits(rows):
        n = rows.shape[0]
        ws = torch.full((n, E), float("nan"), device="cuda")
        idx, w = torch.empty((n, k), dtype=torch.int32, device="cuda"), torch.empty((n, k), dtype=torch.float16, device="cuda")
        mx.ops._call("mx_moe_router", rows.data_ptr(), Wt.data_ptr(), idx.data_ptr(), w.data_ptr(), n, H, E, k, ws.data_ptr())
        return host(ws), host(idx), host(w)

    Wt, xt = dev(Wg), dev(x).half()
    got, ids, w = logits(xt)
    ref = router_logits(x, Wg)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), "logits: %d of %d differ" % ((got != ref).sum(), ref.size)
    shifted = flat[4:].reshape(T, H)
    assert shifted.data_ptr() % 16 == 8
    for a, b in zip(logits(shifted), (got, ids, w)):
        assert np.array_equal(a, b)
    for a, b in zip(logits(xt[T - 1:].clone()), (got, ids, w)):
        assert np.array_equal(a[0], b[T - 1])


@pytest.mark.parametrize("T,E,k,H", [(16, 33, 5, 1040), (40, 65, 4, 16), (300, 33, 5, 36), (250, 33, 5, 1056), (333, 128, 8, 2048), (1030, 257, 8, 288), (2050, 60, 6, 544)])
def test_moe_router_token_tiles(mx, T, E, k, H):
    """Picks against logits summed in 64 bits, over the tile sizes.  A pick may differ only where two logits are within 4e-6: the fp32 sums of up to 2048
    products are off by 6e-7 each (weights of 1 / sqrt(H)), and a probability carries (max - logit) * 2^-23 of exp, below 2e-6 here.
    Neighbours at the edge of the top k are about 0.05 apart, so fewer than one token in a thousand can differ."""
    x = f16(O.normal(9150 + T, (T, H)))
    Wg = O.normal(9151 + E, (E, H), 0.0, 1.0 / np.sqrt(H)).astype(np.float32)
    idx, w = mx.ops.moe_router(dev(x).half(), dev(Wg), E, k)
    logits = (x.astype(np.float64) @ Wg.astype(np.float64).T).astype(np.float32)
    ids_ref, w_ref = O.route_from_logits(logits, k)
    idx_h = host(idx)
    same = (idx_h == ids_ref).all(axis=1)
    for t in np.where(~same)[0]:
        a, b = sorted(set(idx_h[t]) - set(ids_ref[t])), sorted(set(ids_ref[t]) - set(idx_h[t]))
        assert len(a) == len(b) == len(set(a)) and np.abs(logits[t, a] - logits[t, b]).max() <= 4e-6, "differs beyond a tie"
    assert (~same).sum() <= T // 1000
    check(host(w).astype(np.float32)[same], w_ref[same], "router weights", max_rel=2e-3)


@pytest.mark.parametrize("T,E,k", [(5, 64, 64), (3, 65, 2), (9, 129, 8), (2, 257, 8), (4, 1, 1), (6, 1000, 64)])
def test_moe_topk_expert_counts(mx, T, E, k):
    """Experts per lane 1, 2, 4 and 16, every expert picked, one expert only."""
    logits = f16(O.normal(9250 + E, (T, E), 0.0, 2.0))
    idx, w = mx.ops.moe_topk_from_logits(dev(logits).half(), k)
    ids_ref, w_ref = O.route_from_logits(logits, k)
    idx_h = host(idx)
    for t in range(T):
        a, b = set(idx_h[t]) - set(ids_ref[t]), set(ids_ref[t]) - set(idx_h[t])
        assert len(a) == len(b) and sorted(logits[t, list(a)]) == sorted(logits[t, list(b)]), "differs beyond an exact tie"
    assert (np.diff(idx_h, axis=1) > 0).all() if k > 1 else True
    same = (idx_h == ids_ref).all(axis=1)
    check(host(w).astype(np.float32)[same], w_ref[same], "topk weights", max_rel=2e-3)


@pytest.mark.parametrize("T,E,K", [(1, 1, 1), (7, 3, 9), (64, 1024, 1), (65, 1000, 4), (513, 7, 4), (1025, 128, 2), (9000, 1024, 4), (20001, 60, 4), (300, 1100, 3),
                                   (129, 129, 2), (1024, 131, 16), (4096, 128, 4), (4097, 128, 4), (66000, 130, 1)])
def test_moe_packing_device_sizes(mx, T, E, K):
    """Slot counts around the waves' 64-slot pieces and around 4 and 16 slots a lane, one expert, 128 experts and one more, a last
    workgroup with fewer than four, more slots than 2^16; every id drawn freely (a token may name an expert twice)."""
    rng = np.random.default_rng(T * E)
    ids = np.minimum(rng.integers(0, E, (T, K)), rng.integers(0, E, (T, K))).astype(np.int32)
    w = f16(rng.random((T, K)).astype(np.float32))
    off_r, si_r, wp_r, t2p_r = O.build_moe_packing(ids, w, E)
    off, si, wp, t2p = mx.ops.moe_build_packing_device(dev(ids), dev(w).half(), E)
    assert np.array_equal(host(off).view(np.uint32), off_r)
    assert np.array_equal(host(si), si_r)
    assert np.array_equal(host(t2p), t2p_r)
    assert np.array_equal(host(wp).astype(np.float32), wp_r)


@pytest.mark.parametrize("E", [7, 128, 129, 131, 1000])
@pytest.mark.parametrize("T,K", [(32, 2), (1000, 4), (1900, 8), (2500, 8)])
def test_moe_packing_leaves_out_slots_without_an_expert(mx, T, K, E):
    """Ids below 0 and from E on, among them those that a last workgroup of fewer than four experts counts next to its own (E to E + 2), with 4, 16
    and more slots a lane: such slots reach no expert's rows, and nothing is written for them or behind the last row."""
    rng = np.random.default_rng(T + E)
    ids = rng.integers(0, E, (T, K)).astype(np.int32)
    odd = rng.random((T, K)) < 0.3
    ids[odd] = rng.choice(np.array([-1, -(2 ** 31), E, E + 1, E + 2, E + 3, 65536 + E - 1, 2 ** 31 - 1], np.int32), int(odd.sum()))
    w = f16(rng.random((T, K)).astype(np.float32))
    flat = ids.ravel()
    kept = np.flatnonzero((flat >= 0) & (flat < E))
    order = kept[np.argsort(flat[kept], kind="stable")]
    n = len(order)
    off = torch.full((E + 2,), 77, dtype=torch.int32, device="cuda")
    si, t2p = (torch.full((T * K,), -77, dtype=torch.int32, device="cuda") for _ in range(2))
    wp = torch.full((T * K,), -7.0, dtype=torch.float16, device="cuda")
    ids_d, w_d = dev(ids), dev(w).half()
    mx.ops._call("mx_moe_build_packing_device", ids_d.data_ptr(), w_d.data_ptr(), T, K, E, off.data_ptr(), si.data_ptr(), wp.data_ptr(), t2p.data_ptr())
    assert np.array_equal(host(off), np.append(np.concatenate([[0], np.cumsum(np.bincount(flat[kept], minlength=E))]), 77))
    assert np.array_equal(host(si)[:n], order // K) and np.array_equal(host(wp).astype(np.float32)[:n], w.ravel()[order])
    place = np.full(T * K, -77)
    place[order] = np.arange(n)
    assert np.array_equal(host(t2p), place)
    assert (host(si)[n:] == -77).all() and (host(wp)[n:] == -7.0).all()


@pytest.mark.parametrize("T,K,H", [(1, 4, 2880), (3, 5, 8), (2, 9, 20), (33, 8, 1032), (64, 8, 2048), (130, 9, 1032), (127, 5, 1032),
                                   (5, 1, 16), (9, 2, 40), (9, 3, 40), (4, 6, 64), (4, 7, 64), (4, 16, 64), (3, 17, 64)])
def test_moe_reduce_columns(mx, T, K, H):
    """Rows of whole 8-column pieces and not, slot counts at and around the two, four, six and eight rows requested at once, in one group and
    several: fp32 sums of the fp16 rows in slot order."""
    rng = np.random.default_rng(H)
    packed = f16(O.normal(9600, (T * K, H)))
    rows = rng.permutation(T * K).astype(np.int32)
    w = f16(rng.random(T * K).astype(np.float32))
    y0 = f16(O.normal(9601, (T, H)))
    s, a = np.zeros((T, H), np.float32), y0.astype(np.float32).copy()
    for k in range(K):
        r = rows.reshape(T, K)[:, k]
        s += packed[r].astype(np.float32)
        a = (a.astype(np.float64) + w[r, None].astype(np.float64) * packed[r].astype(np.float64)).astype(np.float32)   # one rounding per term (fma)
    y = mx.ops.moe_prefill_reduce_sum(dev(packed).half(), dev(rows), T, K, H)
    assert np.array_equal(host(y).astype(np.float32), f16(s))
    ya = mx.ops.moe_prefill_reduce(dev(packed).half(), dev(rows), dev(w).half(), dev(y0).half(), T, K, H)
    d = np.abs(host(ya).astype(np.float32) - f16(a))
    assert (d <= np.maximum(np.abs(a), 2.0 ** -14) * 2.0 ** -10).all()   # one fp16 unit in the last place: fma or multiply and add


def ref_q8_of(y_half):
    return O.quantize_q8_1(y_half.astype(np.float32))


@pytest.mark.parametrize("rows,hidden", [(1, 4096), (3, 2880), (17, 128), (2, 8192)])
def test_rms_norm_f32w_q8(mx, rows, hidden):
    x = f16(O.normal(9300, (rows, hidden)))
    w = (1.0 + O.normal(9301, (hidden,), 0.0, 0.1)).astype(np.float32)
    eps = 1e-6
    y, q8 = mx.ops.rms_norm_f32w_q8(dev(x).half(), dev(w), eps)
    y_h = host(y)
    xd = x.astype(np.float64)
    ref = xd / np.sqrt((xd * xd).mean(axis=1, keepdims=True) + eps) * w.astype(np.float64)
    check(y_h.astype(np.float32), ref, "rms_norm_f32w_q8 y", max_rel=1.5e-3)   # 1 fp16 ulp + rsqrt
    assert np.array_equal(host(q8), ref_q8_of(y_h).reshape(-1)), "q8 stream == quantize_q8_1(y)"
    assert np.array_equal(host(q8), host(mx.ops.quantize_q8_1(y))), "q8 stream == the standalone quantizer on y"


@pytest.mark.parametrize("rows,hidden", [(32, 128), (5, 256), (1, 4096)])
def test_gated_rms_norm_q8(mx, rows, hidden):
    x = O.normal(9400, (rows, hidden)).astype(np.float32)
    z = f16(O.normal(9401, (rows, hidden)))
    w = f16(1.0 + O.normal(9402, (hidden,), 0.0, 0.1))
    eps = 1e-6
    y, q8 = mx.ops.gated_rms_norm_q8(dev(x), dev(z).half(), dev(w).half(), eps)
    y_h = host(y)
    xd, zd = x.astype(np.float64), z.astype(np.float64)
    ref = w.astype(np.float64) * (xd / np.sqrt((xd * xd).mean(axis=1, keepdims=True) + eps)) * (zd / (1.0 + np.exp(-zd)))
    check(y_h.astype(np.float32), ref, "gated_rms_norm_q8 y", max_rel=1.5e-3)
    assert np.array_equal(host(q8), ref_q8_of(y_h).reshape(-1))


@pytest.mark.parametrize("n", [32, 2880 * 4, 768 * 131])
@pytest.mark.parametrize("oai", [False, True])
def test_swiglu_q8(mx, n, oai):
    """swiglu / swiglu_oai (src/ops/elementwise.cpp:449-492) with the fused block_q8_1x emitter: y against the
    closed form in fp64, the stream bit-identical to quantize_q8_1 of the rounded y."""
    g = f16(O.normal(9500 + n, (n,), 0.0, 3.0))        # sigma 3: the OAI clamp at 7 is exercised
    u = f16(O.normal(9501 + n, (n,), 0.0, 3.0))
    y, q8 = mx.ops.swiglu_q8(dev(g).half(), dev(u).half(), oai=oai)
    y_h = host(y)
    gd, ud = g.astype(np.float64), u.astype(np.float64)
    if oai:
        x, z = np.minimum(gd, 7.0), np.clip(ud, -7.0, 7.0)
        ref = x / (1.0 + np.exp(-1.702 * x)) * (z + 1.0)
    else:
        ref = gd / (1.0 + np.exp(-gd)) * ud
    check(y_h.astype(np.float32), ref, "swiglu%s y" % ("_oai" if oai else ""), max_rel=1.5e-3)
    assert np.array_equal(host(q8), ref_q8_of(y_h).reshape(-1)), "q8 stream == quantize_q8_1(y)"
    _, q8_only = mx.ops.swiglu_q8(dev(g).half(), dev(u).half(), oai=oai, want_y=False)
    assert torch.equal(q8_only, q8)


@pytest.mark.parametrize("n", [32, 64, 1024, 2048 + 96, 32 * 1001, 524288 - 32, 524288, 524288 + 96])
def test_q8_producers_on_8_and_16_byte_boundaries(mx, n):
    """Eight elements per thread on 16-byte boundaries (SwiGLU: from 524288 elements on), four on 8-byte ones: the same fp16 values and q8 bytes (both evaluate one
    element alike), at sizes that end inside a workgroup, against the quantizer of the oracle; halves, a signed zero and an infinity among them."""
    g, u = f16(O.normal(9600 + n, (n + 4,), 0.0, 3.0)), f16(O.normal(9601 + n, (n + 4,)))
    g[5:12] = [127.0, 0.5, -0.5, 2.5, -2.5, 1.5, -0.0]
    tg, tu = dev(g).half(), dev(u).half()
    x8, x16 = tg[4:], tg[4:].clone()
    assert x8.data_ptr() % 16 == 8 and x16.data_ptr() % 16 == 0
    for quantize, oracle in ((mx.ops.quantize_q8_1, O.quantize_q8_1), (mx.ops.quantize_q8_1s, O.quantize_q8_1s)):
        ref = oracle(g[4:])
        assert np.array_equal(host(quantize(x8)).reshape(-1), ref.reshape(-1)) and np.array_equal(host(quantize(x16)).reshape(-1), ref.reshape(-1))
    for oai in (False, True):
        y8, q8 = mx.ops.swiglu_q8(x8, tu[4:], oai=oai)
        y16, q16 = mx.ops.swiglu_q8(x16, tu[4:].clone(), oai=oai)
        assert torch.equal(y8, y16) and torch.equal(q8, q16)
        assert np.array_equal(host(q16), ref_q8_of(host(y16)).reshape(-1))
    inf = x16.clone()
    inf[3] = float("inf")
    off = torch.empty(n + 4, dtype=torch.float16, device=inf.device)[4:]
    off.copy_(inf)
    assert torch.equal(mx.ops.quantize_q8_1(inf), mx.ops.quantize_q8_1(off))
