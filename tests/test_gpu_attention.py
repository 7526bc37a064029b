"""GPU parity of the attention kernels against the oracle:
gqa_attention over fp16/fp32 ring caches, the fused full-attention decode step
(norms + RoPE + append + attention + gate), paged batched decode and causal
prefill."""
import numpy as np
import pytest
import torch

from gpu_util import assert_close, rel_l2, to_dev, to_host
from workloads import attn_decode_case, f16, prefill_inputs, widen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,D,start,length,cap", [
    (8, 2, 256, 0, 513, 2048),       # 0.8B-shaped
    (16, 4, 256, 1900, 700, 2048),   # ring wrap
    (16, 2, 128, 0, 3000, 4096),     # G = 8
    (4, 4, 64, 3, 1, 16),            # one key
    (2, 2, 64, 10, 64, 64),          # full ring
    (16, 4, 256, 0, 8192, 8192),     # 4B-shaped context
])
@pytest.mark.parametrize("kv16", [True, False])
def test_gqa_attention(anelm, orc, dev, nh, nkv, D, start, length, cap, kv16):
    rng = np.random.default_rng(200 + length)
    q = rng.standard_normal((nh, 2 * D)).astype(np.float32)
    kc16 = f16(rng.standard_normal((cap, nkv, D)))
    vc16 = f16(rng.standard_normal((cap, nkv, D)))
    kc, vc = widen(kc16), widen(vc16)
    want = orc.gqa_attention(q, kc, vc, nh, nkv, D, 2 * D, start, length, cap)
    dk = to_dev(kc16 if kv16 else kc, dev)
    dv = to_dev(vc16 if kv16 else vc, dev)
    got = anelm.ops.gqa_attention(to_dev(q, dev), dk, dv, nh, nkv, D, 2 * D, start, length, cap)
    assert_close(to_host(got), want, what=f"gqa {nh}/{nkv} D{D} len{length}")


def test_gqa_attention_empty_cache(anelm, dev):
    out = torch.full((8, 256), 7.0, device=dev)
    q = torch.zeros(8, 512, device=dev)
    kc = torch.zeros(4, 2, 256, device=dev, dtype=torch.float16)
    anelm.ops.gqa_attention(q, kc, kc, 8, 2, 256, 512, 0, 0, 4, out=out)
    assert torch.all(out == 0)


def _run_decode(anelm, c, dev, rope_mode=0, gate=True, cos_row=None, sin_row=None):
    dk, dv = to_dev(c.k_cache, dev), to_dev(c.v_cache, dev)
    ring = anelm.ops.KVRing(c.capacity, c.start, c.length)
    out = anelm.ops.full_attn_decode(
        to_dev(c.q_gate, dev), to_dev(c.k, dev), to_dev(c.v, dev), dk, dv, to_dev(c.q_norm_w, dev),
        to_dev(c.k_norm_w, dev), ring, c.n_heads, c.n_kv_heads, c.head_dim, c.rot_dim, c.pos,
        c.theta, c.eps, rope_mode, gate, cos_row, sin_row)
    return to_host(out), to_host(dk), to_host(dv), ring.start.value, ring.len.value


def _oracle_decode(orc, c, rope_mode=0, gate=True):
    return orc.full_attn_decode(c.q_gate, c.k, c.v, c.k_cache, c.v_cache, c.q_norm_w, c.k_norm_w,
                                c.n_heads, c.n_kv_heads, c.head_dim, c.rot_dim, c.pos, c.theta,
                                c.eps, rope_mode, gate, c.start, c.length, c.capacity)


def _check_decode(got, want):
    out, kc, vc, st, ln = got
    wo, wk, wv, wst, wln = want
    assert (st, ln) == (wst, wln)
    assert_close(out, wo, what="decode out")
    # the appended rows agree to one fp16 ulp (normalisation sums differ in
    # order); every other slot is untouched
    dk = np.abs(kc.astype(np.int32) - wk.astype(np.int32))
    assert dk.max() <= 1 and np.count_nonzero(dk) <= 8
    assert np.array_equal(vc, wv)


def test_full_attn_decode_08b_step(anelm, orc, dev):
    """0.8B-shaped step: 8 q / 2 kv heads, D 256, 512 cached, position 512."""
    c = attn_decode_case(300)
    _check_decode(_run_decode(anelm, c, dev), _oracle_decode(orc, c))


def test_full_attn_decode_4b_step(anelm, orc, dev):
    """4B-shaped step: 16 q / 4 kv heads over 8191 cached keys -> 8192."""
    c = attn_decode_case(301, n_heads=16, n_kv_heads=4, cached=8191, capacity=8192, pos=8191)
    _check_decode(_run_decode(anelm, c, dev), _oracle_decode(orc, c))


@pytest.mark.parametrize("rope_mode,gate", [(1, True), (0, False), (1, False)])
def test_full_attn_decode_variants(anelm, orc, dev, rope_mode, gate):
    c = attn_decode_case(302 + rope_mode, n_heads=16, n_kv_heads=4, cached=777, capacity=1024,
                         start=900)
    _check_decode(_run_decode(anelm, c, dev, rope_mode, gate), _oracle_decode(orc, c, rope_mode, gate))


@pytest.mark.parametrize("n_heads,n_kv_heads,head_dim,cached", [
    (8, 2, 256, 127),    # G 4 on the matrix cores, 128-key splits: one full split
    (8, 2, 256, 1023),   # 8 splits, merged in the kernel
    (8, 2, 256, 1024),   # 9 splits, the last with one key
    (16, 2, 128, 300),   # G 8, 32-key splits: 10 splits
    (4, 2, 128, 700),    # G 2, 128-key splits (workgroup-wide softmax): 6 splits
    (4, 4, 64, 1000),    # G 1, 256-key splits: 4 splits
])
def test_full_attn_decode_split_merge(anelm, orc, dev, n_heads, n_kv_heads, head_dim, cached):
    """Split records merged in the kernel (up to 16 splits by the last workgroup
    of each kv head) for every head grouping, over a wrapped ring, against the
    oracle."""
    c = attn_decode_case(330 + cached % 97, n_heads=n_heads, n_kv_heads=n_kv_heads, head_dim=head_dim,
                         cached=cached, capacity=cached + 5, start=7)
    _check_decode(_run_decode(anelm, c, dev), _oracle_decode(orc, c))


@pytest.mark.parametrize("cached", [
    127,     # two 64-key splits, the smallest in-kernel merge
    1023,    # 16 splits, the largest merged in the split kernel
    1024,    # 17 splits: the merge kernel
])
def test_full_attn_decode_split_merge_off_alignment(anelm, orc, dev, cached):
    """The same for rings of four query heads per kv head at 4-byte aligned
    addresses, which the vector kernel takes."""
    c = attn_decode_case(330 + cached % 97, n_heads=8, n_kv_heads=2, head_dim=256, cached=cached, capacity=cached + 5,
                         start=7)
    kc, vc = (torch.cat([torch.zeros(2, dtype=torch.float16, device=dev), to_dev(x, dev).flatten()])[2:].view(x.shape)
              for x in (c.k_cache, c.v_cache))
    ring = anelm.ops.KVRing(c.capacity, c.start, c.length)
    out = anelm.ops.full_attn_decode(to_dev(c.q_gate, dev), to_dev(c.k, dev), to_dev(c.v, dev), kc, vc,
                                     to_dev(c.q_norm_w, dev), to_dev(c.k_norm_w, dev), ring, c.n_heads, c.n_kv_heads,
                                     c.head_dim, c.rot_dim, c.pos, c.theta, c.eps)
    _check_decode((to_host(out), to_host(kc), to_host(vc), ring.start.value, ring.len.value), _oracle_decode(orc, c))


@pytest.mark.parametrize("Hq,Hkv,cached,start,rope_mode,rot,gate,scale,off", [
    (8, 2, 0, 0, 0, 64, True, 1.0, 0),          # the new key alone: one wave has a key, seven none
    (16, 4, 15, 3, 1, 64, True, 1.0, 0),        # a whole 16-key block, half-split pairs
    (4, 1, 16, 0, 0, 0, False, 1.0, 0),         # the new key alone in its block; no rotation, no gate
    (16, 4, 127, 100, 1, 96, True, 1.0, 0),     # one full split; pairs that are no multiple of a lane's dims apart
    (8, 2, 128, 7, 0, 64, True, 1.0, 0),        # the new key alone in its split
    (8, 2, 2047, 60, 0, 64, True, 1e-4, 0),     # 16 splits, merged in the kernel; tiny rows
    (8, 2, 2048, 60, 0, 64, True, 3e4, 0),      # 17 splits: the merge kernel; rows past fp16's range
    (16, 4, 16500, 900, 0, 64, True, 1.0, 0),   # three rounds of blocks per wave, a part-filled last one
    (16, 4, 300, 9, 0, 64, True, 1.0, 2),       # rows at 4-byte aligned addresses: the vector kernel
])
def test_full_attn_decode_matrix_core_ring(anelm, dev, Hq, Hkv, cached, start, rope_mode, rot, gate, scale, off):
    """fp16 rings of head_dim 256 with 4 query heads per kv head, at the edges
    of the kernel's blocks, splits and merges, every unused ring slot NaN.
    Against float64 over the same fp16 keys: the fp32 query and weights enter
    the products whole (three fp16 terms each), so the error is that of fp32
    sums of 256 products and of the weights' exponential, 2^-24 * 16 * |score|
    at the scores met here: relative 1e-5.  Without norm weights, so `scale`
    is the rows' scale; large rows make one weight 1 and the output a value."""
    D, cap = 256, cached + 9
    c = attn_decode_case(340 + cached % 89, n_heads=Hq, n_kv_heads=Hkv, cached=cached, capacity=cap, start=start % cap,
                         rot_dim=rot)
    used = (c.start + np.arange(cached)) % cap
    free = np.setdiff1d(np.arange(cap), used)
    c.k_cache[free] = c.v_cache[free] = 0x7e00
    c.q_gate[:, :D] *= scale
    kc, vc = (torch.cat([torch.zeros(off, dtype=torch.float16, device=dev), to_dev(x, dev).flatten()])
              [off:].view(x.shape) for x in (c.k_cache, c.v_cache))
    ring = anelm.ops.KVRing(cap, c.start, cached)
    # the rotation's fp32 cos and sin are given, so both sides use the same
    ang = float(c.pos) * c.theta ** (-np.arange(0, rot, 2) / max(rot, 1))
    cs, sn = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
    out = anelm.ops.full_attn_decode(to_dev(c.q_gate, dev), to_dev(c.k, dev), to_dev(c.v, dev), kc, vc, None, None, ring,
                                     Hq, Hkv, D, rot, c.pos, c.theta, c.eps, rope_mode, gate, cs if rot else None,
                                     sn if rot else None)

    def rotate(x):
        x = x.astype(np.float64).copy()
        a, b = (x[:, 0:rot:2], x[:, 1:rot:2]) if rope_mode == 0 else (x[:, :rot // 2], x[:, rot // 2:rot])
        a, b = a * cs - b * sn, a * sn + b * cs   # (float64 products of the fp32 rows)
        if rope_mode == 0:
            x[:, 0:rot:2], x[:, 1:rot:2] = a, b
        else:
            x[:, :rot // 2], x[:, rot // 2:rot] = a, b
        return x

    slots = np.append(used, (c.start + cached) % cap)
    gk, gv = widen(to_host(kc))[slots].astype(np.float64), widen(to_host(vc))[slots].astype(np.float64)
    assert_close(gk[-1].astype(np.float32), rotate(c.k).astype(np.float32), rel=1e-3, max_abs=4e-3, what="new key")
    assert np.array_equal(to_host(vc)[slots[-1]], f16(c.v))
    q = rotate(c.q_gate[:, :D])
    got = to_host(out)
    for h in range(Hq):
        s = gk[:, h * Hkv // Hq] @ q[h] / 16.0
        p = np.exp(s - s.max())
        want = (p / p.sum()) @ gv[:, h * Hkv // Hq]
        if gate:
            want = want / (1.0 + np.exp(-c.q_gate[h, D:].astype(np.float64)))
        err = np.linalg.norm(got[h] - want) / np.linalg.norm(want)
        tol = max(1e-5, 2.0 ** -24 * 16 * np.abs(s).max())
        assert err <= tol, (h, err, tol)


@pytest.mark.parametrize("cached", [0, 40, 111, 128])
def test_full_attn_decode_idle_waves(anelm, dev, cached):
    """Splits with fewer 16-key blocks than waves: the waves without a block
    load the last key's slot too (here still unwritten, every pair of its
    halves a NaN as fp32, which a weight of 0 would not silence) over the LDS
    that they then give their empty rows in; those loads have landed by then."""
    c = attn_decode_case(360 + cached, n_heads=4, n_kv_heads=1, cached=cached, capacity=256, start=0)

    def step():
        return to_host(anelm.ops.full_attn_decode(
            to_dev(c.q_gate, dev), to_dev(c.k, dev), to_dev(c.v, dev), to_dev(c.k_cache, dev), to_dev(c.v_cache, dev),
            to_dev(c.q_norm_w, dev), to_dev(c.k_norm_w, dev), anelm.ops.KVRing(c.capacity, c.start, c.length),
            c.n_heads, c.n_kv_heads, c.head_dim, c.rot_dim, c.pos, c.theta, c.eps))

    clean = step()
    c.v_cache[cached:] = 0x7fff
    assert np.array_equal(step(), clean)


@pytest.mark.parametrize("what", ["v", "v_last", "v_new", "k_masked", "k_nan"])
@pytest.mark.parametrize("cached", [20, 700, 9000])
def test_full_attn_decode_infinite_rows(anelm, dev, what, cached):
    """Infinities among the ring's used keys (values past fp16's range) give
    what fp32 products give: an infinite value makes its output dim infinite, a
    key whose score is -inf weighs nothing, a NaN key makes every head of its
    kv head NaN -- and nothing else changes.  Query rows of one sign in dim 0,
    where the infinite key element is, so all four heads score it -inf."""
    D, Hq, Hkv, cap = 256, 8, 2, cached + 9
    c = attn_decode_case(370 + cached % 89, n_heads=Hq, n_kv_heads=Hkv, cached=cached, capacity=cap, start=cap // 3,
                         rot_dim=0)
    used = (c.start + np.arange(cached)) % cap
    c.q_gate[:, 0] = np.abs(c.q_gate[:, 0]) + 0.1
    inf, slot = np.uint16(0x7c00), used[cached // 2]
    if what == "v":
        c.v_cache[slot, 0, 17] = inf
    elif what == "v_last":
        c.v_cache[used[-1], 0, 17] = inf
    elif what == "v_new":
        c.v[0, 17] = 1e5
    elif what == "k_masked":
        c.k_cache[slot, 0, 0] = inf | 0x8000
    else:
        c.k_cache[slot, 0, 5] = 0x7e00
    kc, vc = to_dev(c.k_cache, dev), to_dev(c.v_cache, dev)
    ring = anelm.ops.KVRing(cap, c.start, cached)
    got = to_host(anelm.ops.full_attn_decode(to_dev(c.q_gate, dev), to_dev(c.k, dev), to_dev(c.v, dev), kc, vc, None,
                                             None, ring, Hq, Hkv, D, 0, c.pos, c.theta, c.eps)).reshape(Hq, D)
    slots = np.append(used, (c.start + cached) % cap)
    kk, vv = widen(to_host(kc))[slots].astype(np.float64), widen(to_host(vc))[slots].astype(np.float64)
    for h in range(Hq):
        with np.errstate(invalid="ignore"):
            s = kk[:, h * Hkv // Hq] @ c.q_gate[h, :D].astype(np.float64) / 16.0
            p = np.exp(s - s.max())
            v = np.where((p == 0)[:, None], 0.0, vv[:, h * Hkv // Hq])
            want = (p / p.sum()) @ v / (1.0 + np.exp(-c.q_gate[h, D:].astype(np.float64)))
        fin = np.isfinite(want)
        assert np.array_equal(np.isnan(got[h]), np.isnan(want)), (what, h)
        assert np.array_equal(got[h][np.isinf(want)], want[np.isinf(want)]), (what, h)
        if fin.any():
            assert rel_l2(got[h][fin], want[fin]) <= 1e-5, (what, h)


@pytest.mark.parametrize("cached", [60, 1000])
def test_full_attn_decode_small_elements(anelm, dev, cached):
    """Query elements and weights far below their row's largest keep fp32's bits:
    one query element 2^24 times the others over keys that are 0 there, and one
    key scoring 20 above the others over values that are 0 there."""
    D, cap = 256, cached + 9
    c = attn_decode_case(380, n_heads=4, n_kv_heads=1, cached=cached, capacity=cap, start=0, rot_dim=0)
    c.q_gate[:, 3] = 2.0 ** 24
    c.q_gate[:, 0] = 8.0
    c.k_cache[:cached, :, 3] = 0
    c.k_cache[:cached, :, 0] = f16(np.zeros((cached, 1), np.float32))
    c.k_cache[cached // 2, 0, 0] = f16(np.array([40.0], np.float32))[0]
    c.v_cache[cached // 2] = 0
    c.k[:, 3] = c.k[:, 0] = 0
    kc, vc = to_dev(c.k_cache, dev), to_dev(c.v_cache, dev)
    got = to_host(anelm.ops.full_attn_decode(to_dev(c.q_gate, dev), to_dev(c.k, dev), to_dev(c.v, dev), kc, vc, None,
                                             None, anelm.ops.KVRing(cap, 0, cached), 4, 1, D, 0, c.pos, c.theta,
                                             c.eps, gate=False)).reshape(4, D)
    kk, vv = widen(to_host(kc))[:cached + 1, 0].astype(np.float64), widen(to_host(vc))[:cached + 1, 0].astype(np.float64)
    for h in range(4):
        s = kk @ c.q_gate[h, :D].astype(np.float64) / 16.0
        p = np.exp(s - s.max())
        want = (p / p.sum()) @ vv
        # fp32 sums of 256 products, the weights' exponential at |score| up to 25
        assert rel_l2(got[h], want) <= 2.0 ** -24 * 16 * np.abs(s).max(), h


def test_full_attn_decode_table_row(anelm, orc, dev):
    """cos/sin passed as the reference's table row give the same step."""
    c = attn_decode_case(305)
    cs, sn = orc.rope_table(c.pos + 1, c.rot_dim, c.theta)
    _check_decode(_run_decode(anelm, c, dev, cos_row=cs[c.pos], sin_row=sn[c.pos]),
                  _oracle_decode(orc, c))


def test_full_attn_decode_consecutive_steps_wrap_ring(anelm, orc, dev):
    """Five steps through a small full ring: slots are overwritten oldest first."""
    rng = np.random.default_rng(306)
    c = attn_decode_case(306, n_heads=8, n_kv_heads=2, cached=30, capacity=32, start=0)
    dk, dv = to_dev(c.k_cache, dev), to_dev(c.v_cache, dev)
    ring = anelm.ops.KVRing(c.capacity, c.start, c.length)
    kc, vc, st, ln = c.k_cache, c.v_cache, c.start, c.length
    qn, kn = to_dev(c.q_norm_w, dev), to_dev(c.k_norm_w, dev)
    for step in range(5):
        qg = rng.standard_normal((8, 512)).astype(np.float32)
        k = rng.standard_normal((2, 256)).astype(np.float32)
        v = rng.standard_normal((2, 256)).astype(np.float32)
        pos = 30 + step
        out = anelm.ops.full_attn_decode(to_dev(qg, dev), to_dev(k, dev), to_dev(v, dev), dk, dv,
                                         qn, kn, ring, 8, 2, 256, 64, pos)
        wo, kc, vc, st, ln = orc.full_attn_decode(qg, k, v, kc, vc, c.q_norm_w, c.k_norm_w, 8, 2,
                                                  256, 64, pos, 1e7, 1e-6, 0, True, st, ln, 32)
        assert (ring.start.value, ring.len.value) == (st, ln)
        assert_close(to_host(out), wo, what=f"step {step}")
        kc = to_host(dk)   # continue from the device cache (fp16 ulp differences stay local)
    assert (st, ln) == (3, 32)


@pytest.mark.parametrize("nh,nkv,D,P", [(16, 4, 256, 16), (16, 2, 128, 5), (4, 4, 64, 32), (8, 1, 128, 1)])
def test_paged_decode(anelm, orc, dev, nh, nkv, D, P):
    """Ragged sequences over shuffled pages (lengths cross the split sizes of
    every head grouping; page sizes that do and do not divide a split)."""
    rng = np.random.default_rng(307 + P)
    n_seqs = 6
    lens = np.array([1, 17, 300, 1024, 2049, 0], np.int32)
    max_len = 2049
    max_pages = (max_len + P - 1) // P
    n_pages = int(sum((l + P - 1) // P for l in lens)) + 3
    perm = rng.permutation(n_pages)
    table = np.zeros((n_seqs, max_pages), np.int32)
    kp16 = f16(rng.standard_normal((n_pages, nkv, P, D)))
    vp16 = f16(rng.standard_normal((n_pages, nkv, P, D)))
    q = rng.standard_normal((n_seqs, nh, D)).astype(np.float32)
    used = 0
    for s, l in enumerate(lens):
        npg = (l + P - 1) // P
        table[s, :npg] = perm[used:used + npg]
        used += npg
    got = to_host(anelm.ops.attn_decode_paged(
        to_dev(q, dev), to_dev(kp16, dev), to_dev(vp16, dev), to_dev(table, dev), to_dev(lens, dev),
        max_len, nh, nkv, D, P))
    for s, l in enumerate(lens):
        if l == 0:
            assert np.all(got[s] == 0)
            continue
        pages = table[s, :(l + P - 1) // P]
        kc = widen(kp16[pages]).transpose(0, 2, 1, 3).reshape(-1, nkv, D)[:l]
        vc = widen(vp16[pages]).transpose(0, 2, 1, 3).reshape(-1, nkv, D)[:l]
        want = orc.gqa_attention(q[s], kc, vc, nh, nkv, D, D, 0, l, l)
        assert_close(got[s], want, what=f"seq {s} len {l}")


# ---------------------------------------------------------------- prefill
@pytest.mark.parametrize("S,Hq,Hkv,D", [(100, 4, 1, 256), (77, 8, 2, 128), (64, 2, 2, 256),
                                        (130, 16, 2, 128), (1, 4, 1, 256), (95, 8, 2, 256),
                                        (257, 16, 4, 256)])
def test_prefill_small(anelm, orc, dev, S, Hq, Hkv, D):
    q, k, v = prefill_inputs(400 + S, S, Hq, Hkv, D)
    got = to_host(anelm.ops.attn_prefill(to_dev(q, dev), to_dev(k, dev), to_dev(v, dev)))
    assert_close(got, orc.prefill_attention(q, k, v), what=f"prefill S{S} {Hq}/{Hkv} D{D}")


def test_prefill_4096_rows(anelm, orc, dev):
    """Causal prefill at S=4096, 16 q / 4 kv heads, D 256: sampled rows vs the
    oracle (the oracle runs each row as a decode call over keys 0..t)."""
    S, Hq, Hkv, D = 4096, 16, 4, 256
    q, k, v = prefill_inputs(401, S, Hq, Hkv, D)
    out = anelm.ops.attn_prefill(to_dev(q, dev), to_dev(k, dev), to_dev(v, dev))
    got = to_host(out)
    rows = [0, 1, 31, 32, 33, 63, 64, 127, 128, 1000, 2047, 2048, 3071, 4094, 4095]
    rows += list(np.random.default_rng(402).integers(0, S, 5))
    for t in rows:
        want = orc.prefill_attention(q, k, v, int(t), int(t) + 1)[0]
        assert_close(got[t], want, what=f"row {t}")
    # fp16 output variant: same values rounded
    got16 = widen(to_host(anelm.ops.attn_prefill(to_dev(q, dev), to_dev(k, dev), to_dev(v, dev),
                                                 torch.float16)))
    assert_close(got16, got, what="fp16 output")


@pytest.mark.parametrize("S,Hq,Hkv", [
    (700, 4, 1),      # 16-token groups, six key parts merged by the second kernel
    (1700, 8, 2),     # 32-token groups, three parts, only the long groups cut
    (5800, 16, 4),    # 64-token groups, one wave per group of 8 tokens, a ragged last one
])
def test_prefill_cuts_both_outputs(anelm, orc, dev, S, Hq, Hkv):
    """The bare core in each of its cuts: sampled rows against the oracle, and
    fp16 rows that are the fp32 rows rounded."""
    q, k, v = prefill_inputs(410 + S, S, Hq, Hkv, 256)
    args = [to_dev(x, dev) for x in (q, k, v)]
    got = to_host(anelm.ops.attn_prefill(*args))
    for t in [0, 7, 8, 31, 32, 63, 64, S // 2, S - 41, S - 1]:
        assert_close(got[t], orc.prefill_attention(q, k, v, t, t + 1)[0], what=f"row {t}")
    assert np.array_equal(to_host(anelm.ops.attn_prefill(*args, torch.float16)), f16(got))


def test_prefill_repeated_calls_are_identical(anelm, orc, dev):
    """Key parts leave records in scratch that the next call writes over:
    back-to-back calls of different sizes and cuts give bit-identical rows, and
    match the oracle."""
    runs = {}
    for S in (700, 130, 700, 64, 700):
        q, k, v = prefill_inputs(990 + S, S, 16, 4, 256)
        got = to_host(anelm.ops.attn_prefill(to_dev(q, dev), to_dev(k, dev), to_dev(v, dev)))
        if S in runs:
            assert np.array_equal(got, runs[S]), f"S={S}: repeated call differs"
        else:
            runs[S] = got
            for t in (0, S // 3, S - 1):
                assert_close(got[t], orc.prefill_attention(q, k, v, t, t + 1)[0], what=f"S{S} row {t}")


def test_full_attn_decode_without_norms(anelm, orc, dev):
    """q/k arriving normalised (scripts/serve_hybrid.py:89-107: half-split RoPE,
    cache append, attention, sigmoid gate, no q/k RMSNorm): NULL norm weights,
    checked against the oracle's RoPE, fp16 append and gqa_attention."""
    c = attn_decode_case(321, n_heads=16, n_kv_heads=4, head_dim=256, cached=300, capacity=4096)
    D, G = c.head_dim, c.n_heads
    dk, dv = to_dev(c.k_cache, dev), to_dev(c.v_cache, dev)
    ring = anelm.ops.KVRing(c.capacity, c.start, c.length)
    out = anelm.ops.full_attn_decode(to_dev(c.q_gate, dev), to_dev(c.k, dev), to_dev(c.v, dev), dk, dv,
                                     None, None, ring, G, c.n_kv_heads, D, c.rot_dim, c.pos, c.theta,
                                     c.eps, rope_mode=1, gate=True)
    q, k = orc.apply_rope(c.q_gate, c.k, G, c.n_kv_heads, D, 2 * D, D, c.rot_dim, c.pos, c.theta, mode=1)
    slot = (c.start + c.length) % c.capacity
    kc, vc = c.k_cache.copy(), c.v_cache.copy()
    kc[slot], vc[slot] = f16(k), f16(c.v)
    want = orc.gqa_attention(q, widen(kc), widen(vc), G, c.n_kv_heads, D, 2 * D, c.start, c.length + 1,
                             c.capacity)
    want = orc.mul_sigmoid(want, c.q_gate[:, D:])
    assert (ring.start.value, ring.len.value) == (c.start, c.length + 1)
    assert_close(to_host(out), want, what="decode without norms")
    assert np.array_equal(to_host(dk)[slot], kc[slot]) and np.array_equal(to_host(dv)[slot], vc[slot])
