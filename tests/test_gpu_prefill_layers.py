"""GPU parity of the prompt prefill through each layer core from its
projections, against the oracle's per-token decode steps (the reference
prefills by running the decode core once per prompt token: generate.cpp:55-85,
models/llm/qwen3_5.cpp:1164-1217):

* anelm_full_attn_prefill == S x orc_full_attn_decode (q/k RMSNorm, RoPE at
  each position, fp16 ring append, attention over the ring after the append,
  sigmoid gate), over a cached prefix in a wrapped ring, with the ring
  overflowing inside the prompt, without norms / gate, and at the prefill
  workload's size (4096 tokens, 16 q / 4 kv heads) on sampled rows;
* anelm_deltanet_prefill_from_proj == S x orc_deltanet_from_proj (conv ring
  + SiLU + split, l2 norm, gates, recurrence, gated norm): outputs, final
  state, conv ring and its position.
"""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import assert_close, to_dev, to_host
from workloads import f16, widen

pytestmark = pytest.mark.gpu


def _attn_case(seed, S, Hq, Hkv, D, cap, start, len0):
    rng = np.random.default_rng(seed)
    kc = np.zeros((cap, Hkv, D), np.uint16)
    vc = np.zeros((cap, Hkv, D), np.uint16)
    slots = (start + np.arange(len0)) % cap
    kc[slots] = f16(rng.standard_normal((len0, Hkv, D)))
    vc[slots] = f16(rng.standard_normal((len0, Hkv, D)))
    return dict(q_gate=rng.standard_normal((S, Hq, 2 * D)).astype(np.float32),
                k=rng.standard_normal((S, Hkv, D)).astype(np.float32),
                v=rng.standard_normal((S, Hkv, D)).astype(np.float32),
                kc=kc, vc=vc,
                qw=(1 + 0.02 * rng.standard_normal(D)).astype(np.float32),
                kw=(1 + 0.02 * rng.standard_normal(D)).astype(np.float32))


def _run_prefill(anelm, dev, c, S, Hq, Hkv, D, rot, cap, start, len0, pos0, norms, rope_mode, gate):
    kc, vc = to_dev(c["kc"], dev), to_dev(c["vc"], dev)
    ring = anelm.ops.KVRing(cap, start, len0)
    tab = anelm.ops.rope_table(rot, pos0 + S, 1e7, dev) if rot else None
    out = anelm.ops.full_attn_prefill(to_dev(c["q_gate"], dev), to_dev(c["k"], dev), to_dev(c["v"], dev), kc, vc,
                                      to_dev(c["qw"], dev) if norms else None,
                                      to_dev(c["kw"], dev) if norms else None, ring, Hq, Hkv, D, rot, pos0,
                                      rope_mode=rope_mode, gate=gate, rope_table=tab,
                                      rope_rows=pos0 + S if rot else 0)
    return to_host(out), to_host(kc), to_host(vc), ring.start.value, ring.len.value


@pytest.mark.parametrize("S,Hq,Hkv,D,cap,start,len0,norms,rope_mode,gate", [
    (200, 16, 4, 256, 2048, 1900, 300, True, 0, True),   # 4B heads, cached prefix over the ring's end
    (300, 16, 4, 256, 256, 100, 200, True, 0, True),     # ring overflows inside the prompt (window)
    (97, 4, 2, 128, 1024, 0, 0, False, 1, False),        # empty cache, no norms, half-split, no gate
    (64, 8, 1, 256, 512, 5, 448, True, 0, True),         # G = 8, prompt fills the ring exactly
])
def test_full_attn_prefill_matches_decode_steps(anelm, orc, dev, S, Hq, Hkv, D, cap, start, len0, norms,
                                                rope_mode, gate):
    rot, pos0 = D // 4, len0 + 7
    c = _attn_case(1700 + S + Hq, S, Hq, Hkv, D, cap, start, len0)
    print(f"full_attn_prefill S{S} {Hq}/{Hkv} D{D} cap{cap} len0 {len0}", flush=True)
    got, gk, gv, gs, gl = _run_prefill(anelm, dev, c, S, Hq, Hkv, D, rot, cap, start, len0, pos0, norms,
                                       rope_mode, gate)
    kc, vc, st, ln = c["kc"], c["vc"], start, len0
    for t in range(S):
        want, kc, vc, st, ln = orc.full_attn_decode(c["q_gate"][t], c["k"][t], c["v"][t], kc, vc,
                                                    c["qw"] if norms else None, c["kw"] if norms else None,
                                                    Hq, Hkv, D, rot, pos0 + t, 1e7, 1e-6, rope_mode, gate,
                                                    st, ln, cap)
        assert_close(got[t], want, what=f"row {t}")
    assert (gs, gl) == (st, ln)
    # the ring holds the same keys (fp16 rows of the same normalised, rotated
    # values; a sum-of-squares order may move one rounding)
    assert_close(widen(gk), widen(kc), rel=1e-3, max_abs=2e-3, what="k ring")
    assert np.array_equal(gv, vc), "v ring"


def test_full_attn_prefill_from_projection_rows(anelm, orc, dev):
    """q_gate, k and v read from the first projection's rows [S][q_gate | k |
    v] (proj_stride) give the same results as packed arrays."""
    S, Hq, Hkv, D, cap, rot = 150, 16, 4, 256, 1024, 64
    c = _attn_case(1760, S, Hq, Hkv, D, cap, 10, 37)
    packed = _run_prefill(anelm, dev, c, S, Hq, Hkv, D, rot, cap, 10, 37, 40, True, 0, True)
    proj = np.concatenate([c["q_gate"].reshape(S, -1), c["k"].reshape(S, -1), c["v"].reshape(S, -1)], axis=1)
    kc, vc = to_dev(c["kc"], dev), to_dev(c["vc"], dev)
    ring = anelm.ops.KVRing(cap, 10, 37)
    tab = anelm.ops.rope_table(rot, 40 + S, 1e7, dev)
    out = anelm.ops.full_attn_prefill(None, None, None, kc, vc, to_dev(c["qw"], dev), to_dev(c["kw"], dev), ring,
                                      Hq, Hkv, D, rot, 40, rope_table=tab, rope_rows=40 + S,
                                      proj=to_dev(proj, dev))
    assert np.array_equal(to_host(out), packed[0])
    assert np.array_equal(to_host(kc), packed[1]) and np.array_equal(to_host(vc), packed[2])
    assert (ring.start.value, ring.len.value) == packed[3:]


def test_full_attn_prefill_4096_rows(anelm, orc, dev):
    """The prefill workload's size through the layer core: 4096 prompt tokens,
    16 q / 4 kv heads, D 256, empty 8192-key ring.  Sampled rows against the
    oracle's composition for row t: q/k RMSNorm + RoPE per token, fp16 keys
    0..t, gqa_attention, sigmoid gate."""
    S, Hq, Hkv, D, cap, rot = 4096, 16, 4, 256, 8192, 64
    c = _attn_case(1750, S, Hq, Hkv, D, cap, 0, 0)
    got, gk, gv, gs, gl = _run_prefill(anelm, dev, c, S, Hq, Hkv, D, rot, cap, 0, 0, 0, True, 0, True)
    assert (gs, gl) == (0, S)
    rows = [0, 1, 63, 64, 1000, 2047, 2048, 4095] + list(np.random.default_rng(1751).integers(0, S, 4))
    top = max(int(t) for t in rows)
    # every key normalised and rotated at its own position, fp16 as cached
    kc = np.zeros((cap, Hkv, D), np.uint16)
    zq = np.zeros((1, 2 * D), np.float32)
    for j in range(top + 1):
        kn = orc.rmsnorm(c["k"][j], c["kw"], 1e-6)
        kc[j] = f16(orc.apply_rope(zq, kn, 1, Hkv, D, 2 * D, D, rot, j, 1e7, mode=0)[1])
    vc = np.zeros((cap, Hkv, D), np.uint16)
    vc[:top + 1] = f16(c["v"][:top + 1])
    assert_close(widen(gk[:top + 1]), widen(kc[:top + 1]), rel=1e-3, max_abs=2e-3, what="k ring")
    assert np.array_equal(gv[:S], vc[:S]), "v ring"
    for t in rows:
        t = int(t)
        qn = orc.rmsnorm(c["q_gate"][t, :, :D], c["qw"], 1e-6)
        qg = np.concatenate([qn, c["q_gate"][t, :, D:]], axis=1)
        qr, _ = orc.apply_rope(qg, np.zeros((Hkv, D), np.float32), Hq, Hkv, D, 2 * D, D, rot, t, 1e7, mode=0)
        att = orc.gqa_attention(qr, widen(kc), widen(vc), Hq, Hkv, D, 2 * D, 0, t + 1, cap)
        want = orc.mul_sigmoid(att, c["q_gate"][t, :, D:])
        assert_close(got[t], want, what=f"row {t}")


@pytest.mark.parametrize("S,Hq,Hkv,cap,start,len0,rope_mode,pad,table_rows,off", [
    (1, 8, 2, 64, 3, 0, 0, 0, 0, 0),              # one token, nothing cached
    (15, 8, 2, 4096, 4090, 4000, 0, 0, 4096, 0),  # part-filled group, many key parts, wrap inside a tile
    (17, 16, 4, 512, 500, 10, 1, 0, 512, 0),      # one token past a group; wrap inside the prompt
    (40, 16, 4, 64, 0, 10, 0, 1, 64, 0),          # rows not 16-byte aligned; a column's first tile wholly masked
    (33, 4, 1, 256, 255, 95, 1, 3, 20, 0),        # one kv head; positions past the RoPE table
    (24, 12, 3, 300, 7, 200, 0, 0, 300, 0),       # kv heads that do not divide the XCDs
    (500, 16, 4, 1024, 600, 300, 0, 0, 1024, 0),  # several key parts of 16-token groups, wrapped ring
    (2100, 16, 4, 4096, 0, 0, 0, 0, 4096, 0),     # more workgroups than compute units
    (5741, 16, 4, 8192, 7000, 70, 0, 0, 6000, 0),  # groups of 64 tokens (one key part), a ragged last one, wrapped ring
    (40, 16, 4, 128, 100, 10, 0, 0, 64, 2),       # a ring at a 4-byte aligned address: gathered
])
def test_full_attn_prefill_cuts(anelm, dev, S, Hq, Hkv, cap, start, len0, rope_mode, pad, table_rows, off):
    """Head_dim 256 with 4 query heads per kv head at the edges of its token
    groups, key tiles and key parts, reading the ring in place.  Against the
    layer's formulas in float64 on the GPU, over q and new keys rounded to fp16
    as the layer keeps them.  Each output row is a weighted mean of values whose
    weights are fp16 (relative 2^-11), so its error is below the usual bar."""
    D, rot, pos0 = 256, 64, len0 + 3
    c = _attn_case(1900 + S + len0, S, Hq, Hkv, D, cap, start, len0)
    stride = Hq * 2 * D + 2 * Hkv * D + pad
    proj = np.zeros((S, stride), np.float32)
    proj[:, :Hq * 2 * D] = c["q_gate"].reshape(S, -1)
    proj[:, Hq * 2 * D:Hq * 2 * D + Hkv * D] = c["k"].reshape(S, -1)
    proj[:, Hq * 2 * D + Hkv * D:Hq * 2 * D + 2 * Hkv * D] = c["v"].reshape(S, -1)
    pd = to_dev(proj, dev)
    kc, vc = (torch.cat([torch.zeros(off, dtype=torch.float16, device=dev), to_dev(c[x], dev).flatten()])[off:]
              .view(c[x].shape) for x in ("kc", "vc"))
    qw, kw = to_dev(c["qw"], dev), to_dev(c["kw"], dev)
    ring = anelm.ops.KVRing(cap, start, len0)
    tab = anelm.ops.rope_table(rot, table_rows, 1e7, dev) if table_rows else None
    out = torch.empty(S, Hq * D, device=dev)
    p = ctypes.c_void_p
    anelm.call("anelm_full_attn_prefill", p(out.data_ptr()), p(pd.data_ptr()),
               p(pd.data_ptr() + 4 * Hq * 2 * D), p(pd.data_ptr() + 4 * (Hq * 2 * D + Hkv * D)), stride,
               p(kc.data_ptr()), p(vc.data_ptr()), p(qw.data_ptr()), p(kw.data_ptr()), S, Hq, Hkv, D, rot, pos0,
               ctypes.c_float(1e7), ctypes.c_float(1e-6), rope_mode, 1, p(tab.data_ptr() if table_rows else None),
               table_rows, ctypes.byref(ring.start), ctypes.byref(ring.len), cap,
               p(torch.cuda.current_stream().cuda_stream))
    assert (ring.start.value, ring.len.value) == (start, len0 + S)

    def rows(x, w, heads):
        x = x.double()
        x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w.double()
        i = torch.arange(0, rot, 2, dtype=torch.float32)
        freq = (1.0 / torch.pow(torch.tensor(1e7), i / rot)).to(dev)
        ang = (torch.arange(pos0, pos0 + S, dtype=torch.float32, device=dev)[:, None] * freq).double()[:, None]
        a, b = (x[..., 0:rot:2], x[..., 1:rot:2]) if rope_mode == 0 else (x[..., :rot // 2], x[..., rot // 2:rot])
        a, b = a * torch.cos(ang) - b * torch.sin(ang), a * torch.sin(ang) + b * torch.cos(ang)
        x = x.clone()
        if rope_mode == 0:
            x[..., 0:rot:2], x[..., 1:rot:2] = a, b
        else:
            x[..., :rot // 2], x[..., rot // 2:rot] = a, b
        return x.float().half()

    slots = (start + torch.arange(len0 + S, device=dev)) % cap
    q = rows(pd[:, :Hq * 2 * D].view(S, Hq, 2 * D)[..., :D], qw, Hq).double()
    want_k, want_v = to_dev(c["kc"], dev).view(torch.float16), to_dev(c["vc"], dev).view(torch.float16)
    want_k[slots[len0:]] = rows(to_dev(c["k"], dev), kw, Hkv)
    want_v[slots[len0:]] = to_dev(c["v"], dev).half()
    got_k = kc.view(torch.float16)
    assert_close(got_k.float().cpu().numpy(), want_k.float().cpu().numpy(), rel=1e-3, max_abs=2e-3, what="k ring")
    assert torch.equal(vc.view(torch.float16), want_v)
    kk, vv = got_k[slots].double(), want_v[slots].double()
    gate = torch.sigmoid(to_dev(c["q_gate"], dev)[..., D:].double())
    mask = torch.arange(len0 + S, device=dev)[None] > len0 + torch.arange(S, device=dev)[:, None]
    for h in range(Hq):
        sc = (q[:, h] @ kk[:, h * Hkv // Hq].t().contiguous() / 16.0).masked_fill(mask, -np.inf)
        want = (torch.softmax(sc, -1) @ vv[:, h * Hkv // Hq].contiguous()) * gate[:, h]
        assert_close(out.view(S, Hq, D)[:, h].cpu().numpy(), want.float().cpu().numpy(), what=f"head {h}")


@pytest.mark.parametrize("S,Hq,Hkv,len0", [
    (24, 8, 2, 0),       # one key part: gated in the kernel
    (24, 8, 2, 3000),    # several: gated in the merge
    (24, 4, 2, 0),       # two query heads per kv head
])
def test_full_attn_prefill_special_gates(anelm, dev, S, Hq, Hkv, len0):
    """Gate logits that are NaN, infinite or past where exp overflows give what
    x / (1 + exp(-g)) gives in fp32: NaN stays NaN, +inf passes the value, -inf
    and anything below -88.8 gives 0.  Against the call without a gate; finite
    logits within the quotient's, the sum's and (2 ulp) exp's rounding."""
    D, cap = 256, 4096
    c = _attn_case(1950 + len0, S, Hq, Hkv, D, cap, 5, len0)
    rng = np.random.default_rng(1951)
    special = np.array([np.nan, np.inf, -np.inf, -100.0, -90.0, -88.0, 88.0, 200.0], np.float32)
    at = rng.integers(0, S * Hq * D, 400)
    c["q_gate"][..., D:].reshape(-1)[:] = 0
    gl = np.ascontiguousarray(c["q_gate"][..., D:]) + (8 * rng.standard_normal((S, Hq, D))).astype(np.float32)
    gl.reshape(-1)[at] = special[np.arange(400) % len(special)]
    c["q_gate"][..., D:] = gl

    def run(gate):
        return _run_prefill(anelm, dev, c, S, Hq, Hkv, D, 64, cap, 5, len0, len0, True, 0, gate)[0]

    plain, got = (run(g).reshape(S, Hq, D).astype(np.float64) for g in (False, True))
    assert np.isfinite(plain).all()
    with np.errstate(over="ignore"):
        # fp32's 1 + exp(-g) is infinite from -88.73 down
        want = np.where(gl < -88.73, 0.0, plain / (1.0 + np.exp(-gl.astype(np.float64))))
    assert np.array_equal(np.isnan(got), np.isnan(gl))
    ok = ~np.isnan(gl)
    assert (np.abs(got - want)[ok] <= 4 * 2.0 ** -23 * np.abs(want)[ok] + 1e-45).all()


@pytest.mark.parametrize("S,Hk,Hv,flags,pos0", [
    (100, 16, 32, 5, 2),      # 4B layer: l2 norm + gated norm, conv ring position 2
    (130, 16, 16, 7, 0),      # 0.8B heads, transformers order
    (2, 16, 32, 5, 1),        # fewer tokens than the ring holds
])
def test_deltanet_prefill_from_proj_matches_decode_steps(anelm, orc, dev, S, Hk, Hv, flags, pos0):
    rng = np.random.default_rng(1800 + S + Hv + flags)
    d, K = 128, 4
    qkv = 2 * Hk * d + Hv * d
    St = (0.1 * rng.standard_normal((Hv, d, d))).astype(np.float32)
    conv_w = (0.5 * rng.standard_normal((qkv, K))).astype(np.float32)
    cs = (0.5 * rng.standard_normal((qkv, K - 1))).astype(np.float32)
    A = np.exp(rng.uniform(0, np.log(16), Hv)).astype(np.float32)
    dtb = rng.standard_normal(Hv).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    proj = rng.standard_normal((S, qkv + Hv * d + 2 * Hv)).astype(np.float32)
    Sd, csd = to_dev(St, dev), to_dev(cs, dev)
    pos = ctypes.c_int(pos0)
    print(f"deltanet_prefill_from_proj S{S} {Hk}k/{Hv}v flags {flags}", flush=True)
    y = to_host(anelm.ops.deltanet_prefill_from_proj(Sd, csd, pos, to_dev(proj, dev), to_dev(conv_w, dev),
                                                     to_dev(A, dev), to_dev(dtb, dev), to_dev(nw, dev), Hk,
                                                     flags, K))
    p = pos0
    for t in range(S):
        yw, St, cs, p = orc.deltanet_from_proj(St, cs, p, proj[t], conv_w, A, dtb, nw, Hk, Hv, K, flags)
        assert_close(y[t], yw, what=f"y token {t}")
    assert pos.value == p
    assert_close(to_host(Sd), St, what="state")
    assert np.array_equal(to_host(csd), cs), "conv ring"


@pytest.mark.parametrize("S,Hk,Hv,flags,pos0,K", [
    (1, 16, 32, 5, 2, 4),      # one token
    (3, 16, 16, 7, 1, 4),      # as many tokens as the conv ring holds
    (63, 2, 4, 5, 0, 4),       # one token short of a chunk
    (64, 2, 2, 7, 2, 4),       # one whole chunk
    (65, 2, 4, 7, 0, 4),       # one token past it
    (2060, 16, 32, 5, 1, 4),   # enough chunks for both value heads of a key head in one workgroup
    (130, 2, 4, 5, 1, 3),      # another conv width: the conv in a pass of its own
    (130, 3, 3, 7, 0, 4),      # rows not 16-byte aligned: likewise
])
def test_deltanet_prefill_from_proj_cuts(anelm, orc, dev, S, Hk, Hv, flags, pos0, K):
    """The prompt pass from projection rows at the edges of its 64-token chunks
    and of its choices, token by token against the decode recurrence (the same
    bars as above; the conv ring holds projection values, bit for bit)."""
    rng = np.random.default_rng(1850 + S + Hv + flags + K)
    d = 128
    qkv = 2 * Hk * d + Hv * d
    St = (0.1 * rng.standard_normal((Hv, d, d))).astype(np.float32)
    conv_w = (0.5 * rng.standard_normal((qkv, K))).astype(np.float32)
    cs = (0.5 * rng.standard_normal((qkv, K - 1))).astype(np.float32)
    A = np.exp(rng.uniform(0, np.log(16), Hv)).astype(np.float32)
    dtb = rng.standard_normal(Hv).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    proj = rng.standard_normal((S, qkv + Hv * d + 2 * Hv)).astype(np.float32)
    Sd, csd = to_dev(St, dev), to_dev(cs, dev)
    pos = ctypes.c_int(pos0)
    y = to_host(anelm.ops.deltanet_prefill_from_proj(Sd, csd, pos, to_dev(proj, dev), to_dev(conv_w, dev),
                                                     to_dev(A, dev), to_dev(dtb, dev), to_dev(nw, dev), Hk,
                                                     flags, K))
    p = pos0
    for t in range(S):
        yw, St, cs, p = orc.deltanet_from_proj(St, cs, p, proj[t], conv_w, A, dtb, nw, Hk, Hv, K, flags)
        assert_close(y[t], yw, what=f"y token {t}")
    assert pos.value == p
    assert_close(to_host(Sd), St, what="state")
    assert np.array_equal(to_host(csd), cs), "conv ring"


@pytest.mark.parametrize("flags,off", [(5, 0), (1, 0), (5, 3 * 128)])
def test_deltanet_prefill_from_proj_over_its_rows(anelm, dev, flags, off):
    """The output may lie over the projection rows: they are read whole first
    (against the call with an output of its own, whose passes round otherwise)."""
    S, Hk, Hv, K, d = 200, 2, 4, 4, 128
    rng = np.random.default_rng(1870 + flags + off)
    qkv, pd = 2 * Hk * d + Hv * d, 2 * Hk * d + 2 * Hv * d + 2 * Hv
    t = {n: to_dev(x.astype(np.float32), dev) for n, x in dict(
        St=0.1 * rng.standard_normal((Hv, d, d)), cs=0.5 * rng.standard_normal((qkv, K - 1)),
        w=0.5 * rng.standard_normal((qkv, K)), A=np.exp(rng.uniform(0, np.log(16), Hv)), dtb=rng.standard_normal(Hv),
        nw=1 + 0.1 * rng.standard_normal(d), proj=rng.standard_normal((S, pd))).items()}

    def run(inside):
        St, cs, proj = t["St"].clone(), t["cs"].clone(), t["proj"].clone()
        y = proj.view(-1)[off:off + S * Hv * d] if inside else torch.empty(S * Hv * d, device=dev)
        pos, p = ctypes.c_int(1), ctypes.c_void_p
        anelm.call("anelm_deltanet_prefill_from_proj", p(y.data_ptr()), p(St.data_ptr()), p(cs.data_ptr()),
                   ctypes.byref(pos), p(proj.data_ptr()), p(t["w"].data_ptr()), p(t["A"].data_ptr()),
                   p(t["dtb"].data_ptr()), p(t["nw"].data_ptr()), S, Hk, Hv, d, d, K, flags,
                   p(torch.cuda.current_stream().cuda_stream))
        return to_host(y.clone()), to_host(St), to_host(cs)

    for got, want, what in zip(run(True), run(False), ("y", "state", "conv ring")):
        assert_close(got, want, rel=1e-5, max_abs=1e-3, what=what)


def test_short_prompt_leaves_captured_decode(anelm, dev):
    """A graph captured from a decode step holds the stream's first buffer (its
    split records); a few tokens behind a long ring on that stream keep the
    records of their key parts elsewhere, so every replay gives the eager step."""
    Hq, Hkv, D, cap = 8, 2, 256, 4096
    c = _attn_case(1990, 1, Hq, Hkv, D, cap, 0, 3000)
    q, k, v = (to_dev(c[n][0], dev) for n in ("q_gate", "k", "v"))
    kc, vc, qw, kw = (to_dev(c[n], dev) for n in ("kc", "vc", "qw", "kw"))
    rng = np.random.default_rng(1991)
    proj = to_dev(rng.standard_normal((100, Hq * 2 * D + 2 * Hkv * D)).astype(np.float32), dev)
    out, s = torch.empty(Hq, D, device=dev), torch.cuda.Stream()

    def step():   # (the same slot each time: a fresh ring object, the position fixed)
        anelm.ops.full_attn_decode(q, k, v, kc, vc, qw, kw, anelm.ops.KVRing(cap, 0, 3000), Hq, Hkv, D, 64, 3000, out=out)

    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        step()
        want = out.clone()
        graph = torch.cuda.CUDAGraph()
        s.synchronize()
        with torch.cuda.graph(graph, stream=s):
            step()
        first = {}
        for tokens in (24, 100, 24):
            got = anelm.ops.full_attn_prefill(None, None, None, kc.clone(), vc.clone(), qw, kw,
                                              anelm.ops.KVRing(cap, 0, 3000), Hq, Hkv, D, 64, 3000, proj=proj[:tokens])
            out.zero_()
            graph.replay()
            s.synchronize()
            assert torch.equal(out, want), tokens
            assert torch.equal(got, first.setdefault(tokens, got.clone()))
    del graph
    anelm.call("anelm_stream_release", ctypes.c_void_p(s.cuda_stream))
