"""Batched decode (model geometry) against the oracle: GQA, ragged lengths, splits, both key formats.

The batched entry point serves the model dispatch sites (src/model/decoder.ts:46-56:
encode_k, compressed_dot, softmax, weighted) for B sequences x KV heads.
Outputs must match the oracle's attention on the same effective K within
|gpu - oracle| <= 1e-5 + 1e-4 |oracle|.
"""
import numpy as np
import pytest

from conftest import REF

pytestmark = pytest.mark.gpu

ATOL, RTOL = 1e-5, 1e-4


def _olayout(oracle, p):
    return oracle.Layout(dim=p.dim, groups=p.groups, row_bytes=p.rowBytes, norm_stride=p.normStride,
                         nibble_dims=p.nibbleDims, max_centroids=p.maxCentroids, perm=p.permutation,
                         group_of=p.groupOf, pos_to_cb=p.positionToCodebook, code_lut=p.codeLut,
                         rotation=p.rotation, centroids=p.centroids, offsets=p.offsets, inv_scales=p.inverseScales)


def _check(out, ref, what):
    err = np.abs(out.astype(np.float64) - ref)
    lim = ATOL + RTOL * np.abs(ref)
    assert np.all(err <= lim), f"{what}: max err {err.max():.3e}, worst ratio {(err / lim).max():.2f}"


def _run(device, oracle, *, params, batch, hq, hkv, dim, lengths, cap, key_format="packed", splits=0, seed=0,
         zero_q=False, pad16=False):
    import torch
    import bgtq
    from bgtq import batched
    batched.bind_torch_stream(device)
    g = torch.Generator().manual_seed(seed)
    k = (torch.randn((batch, hkv, cap, dim), generator=g) * 0.8).half()
    v = torch.randn((batch, hkv, cap, dim), generator=g).half()
    q = torch.randn((batch, hq, dim), generator=g)
    if zero_q:
        q.zero_()
    lengths_t = torch.tensor(lengths, dtype=torch.int32)
    out = torch.empty((batch, hq, dim), dtype=torch.float32, device="cuda")
    kw = {}
    tabs = []
    if key_format == "packed":
        tabs = [bgtq.Tables(device, p) for p in params]
        rb, ns = params[0].rowBytes, params[0].normStride
        pk_len, nm_len = cap * rb + 64, cap * ns + 32
        if pad16:  # 16-byte aligned head and sequence strides
            pk_len, nm_len = (pk_len + 15) // 16 * 16, (nm_len + 7) // 8 * 8
        packed = torch.zeros((batch, hkv, pk_len), dtype=torch.uint8, device="cuda")
        norms = torch.zeros((batch, hkv, nm_len), dtype=torch.int16, device="cuda")
        kd = k.cuda()
        jobs = [dict(tables=tabs[h], src=kd[b, h], src_row_stride=dim, rows=cap, packed=packed[b, h],
                     norms=norms[b, h]) for b in range(batch) for h in range(hkv)]
        batched.encode(device, jobs, "f16")
        kw = dict(tables=tabs, packed=packed, packed_seq_stride=packed.stride(0), packed_head_stride=packed.stride(1),
                  norms=norms, norms_seq_stride=norms.stride(0), norms_head_stride=norms.stride(1))
    else:
        kd = k.cuda()
        kw = dict(k_f16=kd, k_seq_stride=kd.stride(0), k_head_stride=kd.stride(1))
    vd, qd, ld = v.cuda(), q.cuda(), lengths_t.cuda()
    desc = batched.decode_desc(batch=batch, q_heads=hq, kv_heads=hkv, dim=dim, q=qd, out=out, lengths=ld,
                               max_length=max(lengths), v=vd, v_seq_stride=vd.stride(0), v_head_stride=vd.stride(1),
                               splits=splits, **kw)
    ws = torch.zeros(batched.workspace_bytes(desc), dtype=torch.uint8, device="cuda")
    desc = batched.decode_desc(batch=batch, q_heads=hq, kv_heads=hkv, dim=dim, q=qd, out=out, lengths=ld,
                               max_length=max(lengths), v=vd, v_seq_stride=vd.stride(0), v_head_stride=vd.stride(1),
                               splits=splits, workspace=ws, **kw)
    batched.decode(device, desc)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    G = hq // hkv
    refs = {}
    for b in range(batch):
        T = lengths[b]
        for h in range(hkv):
            if key_format == "packed":
                p = params[h]
                pk = packed[b, h, :T * p.rowBytes].cpu().numpy().reshape(T, p.rowBytes)
                nm = norms[b, h, :T * p.normStride].cpu().numpy().view(np.float16).reshape(T, p.normStride)
                keff = oracle.reconstruct(_olayout(oracle, p), oracle.unpack(pk, dim, p.nibbleDims),
                                          nm.astype(np.float32))
            else:
                keff = k[b, h, :T].float().numpy()
            qq = q[b, h * G:(h + 1) * G].numpy()
            _, _, ref = oracle.attention(qq, keff, v[b, h, :T].float().numpy(), np.full(G, T - 1), False)
            refs[(b, h)] = ref
            _check(got[b, h * G:(h + 1) * G], ref.astype(np.float64), f"b{b} kv{h} T={T}")
    for t in tabs:
        t.destroy()
    return got, v, lengths


@pytest.mark.parametrize("dim", [64, 128])
def test_layout_b_gqa_ragged(device, oracle, dim):
    from bgtq import calibrate
    p = calibrate.layout_b(dim)
    print("layout B", dim, flush=True)
    _run(device, oracle, params=[p, p], batch=3, hq=14, hkv=2, dim=dim, lengths=[1, 77, 1000], cap=1000)


@pytest.mark.parametrize("dim", [64, 128])
def test_fp16_keys_baseline(device, oracle, dim):
    print("fp16 K", dim, flush=True)
    _run(device, oracle, params=None, batch=2, hq=14, hkv=2, dim=dim, lengths=[513, 130], cap=600,
         key_format="fp16")


@pytest.mark.parametrize("splits", [1, 3, 7, 12])
def test_forced_splits(device, oracle, splits):
    from bgtq import calibrate
    p = calibrate.layout_b(64)
    print("splits", splits, flush=True)
    _run(device, oracle, params=[p], batch=2, hq=3, hkv=1, dim=64, lengths=[2000, 1500], cap=2000, splits=splits)


@pytest.mark.parametrize("splits", [30, 47])
def test_forced_splits_long(device, oracle, splits):
    """Split merges of every size class: one load round up to 40 splits, two phases beyond."""
    from bgtq import calibrate
    p = calibrate.layout_b(64)
    print("splits", splits, flush=True)
    _run(device, oracle, params=[p], batch=2, hq=7, hkv=1, dim=64, lengths=[6000, 5100], cap=6000, splits=splits)


def test_non_fast_layouts_use_general_kernel(device, oracle):
    """Layouts whose K-steps mix groups (real SmolLM2 heads; layout A) over caches whose strides are no
    multiple of 16 bytes run the general kernel."""
    from bgtq import BlockGTQParameters, calibrate
    m, a = oracle.read_fixture(REF / "model" / "calibration.json")
    heads = [BlockGTQParameters.from_serialized(a[f"h{i}_config"], a[f"h{i}_table"]) for i in (3, 4, 5)]
    rb = max(h.rowBytes for h in heads)
    ns = max(h.normStride for h in heads)
    for h in heads:  # one cache stride for all heads of the layer (src/model/decoder.ts:21 keeps one per head)
        h.rowBytes, h.normStride = rb, ns
    print("smollm2 heads", flush=True)
    _run(device, oracle, params=heads, batch=2, hq=9, hkv=3, dim=64, lengths=[300, 41], cap=300)
    pa = calibrate.layout_a(64)
    print("layout A", flush=True)
    _run(device, oracle, params=[pa, pa], batch=1, hq=14, hkv=2, dim=64, lengths=[700], cap=700)


@pytest.mark.parametrize("dim,splits", [(64, 0), (128, 0), (64, 5), (128, 3)])
def test_layout_a_fused(device, oracle, dim, splits):
    """Layout A (widths 4..8: K-steps spanning two groups; at d=128 nibble and byte codes in one
    K-step and a norm stride of 5) with 16-byte aligned caches: the fused kernel's per-position
    code lookup, ragged GQA batch."""
    from bgtq import calibrate
    p = calibrate.layout_a(dim)
    print("layout A fused", dim, splits, flush=True)
    _run(device, oracle, params=[p, p], batch=3, hq=14, hkv=2, dim=dim, lengths=[1, 77, 2049], cap=2049,
         splits=splits, pad16=True)


@pytest.mark.parametrize("dim,G", [(64, 1), (64, 4), (64, 5), (64, 8), (64, 9), (64, 16), (128, 3), (128, 8),
                                   (128, 12)])
def test_any_layout_group_packing(device, oracle, dim, G):
    """The fused per-position kernel packs four (G <= 4) or two (G <= 8) group slots into one
    matrix-core product and sums them across lanes; G > 8 runs one slot per product. Every
    packing width against the oracle, on layout A (two groups per K-step) and the real heads."""
    from bgtq import calibrate
    p = calibrate.layout_a(dim)
    print("group packing", dim, G, flush=True)
    _run(device, oracle, params=[p, p], batch=2, hq=2 * G, hkv=2, dim=dim, lengths=[300, 1031], cap=1031,
         pad16=True, seed=G)
    if dim == 64:
        heads = _smollm2_heads(oracle, ["h0", "h1", "h22"])
        _run(device, oracle, params=heads, batch=1, hq=3 * G, hkv=3, dim=dim, lengths=[517], cap=517, pad16=True,
             seed=G + 1)


def _smollm2_heads(oracle, names):
    """Reference calibration heads of one layer: one cache row stride and norm stride for all
    (src/model/decoder.ts:21 keeps one per head)."""
    from bgtq import BlockGTQParameters
    m, a = oracle.read_fixture(REF / "model" / "calibration.json")
    heads = [BlockGTQParameters.from_serialized(a[f"{n}_config"], a[f"{n}_table"]) for n in names]
    rb = max(h.rowBytes for h in heads)
    ns = max(h.normStride for h in heads)
    for h in heads:
        h.rowBytes, h.normStride = rb, ns
    return heads


@pytest.mark.parametrize("names,splits", [(("h3", "h56", "h26"), 0), (("h0", "h1", "h22"), 0),
                                          (("h0", "h1", "h22"), 4)])
def test_smollm2_heads_fused(device, oracle, names, splits):
    """Real SmolLM2 calibration heads (K-steps spanning up to four groups, nibble and byte codes in
    one lane's eight positions, 3-6 books, rows of 44 or of an odd 37 bytes, norm strides 4 and 6)
    with 16-byte aligned caches: the fused kernel's per-position code lookup."""
    heads = _smollm2_heads(oracle, names)
    print("smollm2 heads fused", names, splits, flush=True)
    _run(device, oracle, params=heads, batch=2, hq=9, hkv=3, dim=64, lengths=[1000, 77], cap=1000, splits=splits,
         pad16=True)


def test_smollm2_every_layer_fused(device, oracle):
    """All 90 SmolLM2 calibration heads (30 layers x 3 KV heads) through the fused decode."""
    for layer in range(30):
        heads = _smollm2_heads(oracle, [f"h{3 * layer + h}" for h in range(3)])
        print("smollm2 layer", layer, flush=True)
        _run(device, oracle, params=heads, batch=1, hq=9, hkv=3, dim=64, lengths=[150], cap=150, pad16=True,
             seed=layer)


def _widths_1_to_6_d128():
    """d=128, widths 1..6 in six groups: 98 nibble positions (a lane's 8 codes mix nibbles and
    bytes), 79-byte rows (not word aligned), norm stride 6, up to three groups per 32 positions."""
    from bgtq import calibrate
    return calibrate.make_parameters(calibrate.allocate_bits(calibrate.geometric_scores(64), 206, 1, 8))


def test_widths_1_to_6_d128_fused(device, oracle):
    p = _widths_1_to_6_d128()
    assert (p.dim, p.nibbleDims, p.rowBytes, p.normStride) == (128, 98, 79, 6)
    print("widths 1..6 d=128", flush=True)
    _run(device, oracle, params=[p, p], batch=2, hq=14, hkv=2, dim=128, lengths=[77, 1000], cap=1000, pad16=True)


def test_full_context_closed_form(device, oracle):
    """32768-token context: zero q gives the mean of V exactly enough (uniform softmax)."""
    from bgtq import calibrate
    p = calibrate.layout_b(64)
    print("32k zero-q", flush=True)
    got, v, lengths = _run(device, oracle, params=[p, p], batch=2, hq=14, hkv=2, dim=64, lengths=[32768, 32768],
                           cap=32768, zero_q=True)
    for b in range(2):
        for h in range(2):
            mean = v[b, h].float().numpy().astype(np.float64).mean(0)
            _check(got[b, h * 7:(h + 1) * 7], np.broadcast_to(mean, (7, 64)), "mean of V")


def test_full_context_vs_oracle(device, oracle):
    from bgtq import calibrate
    p = calibrate.layout_b(64)
    print("32k random", flush=True)
    _run(device, oracle, params=[p, p], batch=1, hq=14, hkv=2, dim=64, lengths=[32768], cap=32768, seed=5)


def test_optimized_attention_fp16_values_mfma(device, oracle):
    """OptimizedAttention over layout-B packed K and FP16 V (the matrix-core path), inspect() included."""
    import bgtq
    from bgtq import calibrate
    p = calibrate.layout_b(128)
    rng = np.random.default_rng(9)
    T = 4096
    k = rng.standard_normal((T, 128)).astype(np.float16)
    v = rng.standard_normal((T, 128)).astype(np.float16).astype(np.float32)
    q = rng.standard_normal((3, 128)).astype(np.float32)
    keys = bgtq.PackedKeys.create(device, p, T)
    values = bgtq.Values(device, 128, T, dtype="f16")
    att = bgtq.OptimizedAttention.create(device, keys, values, 3)
    try:
        keys.append(k.view(np.uint16))
        values.append(v)
        packed, norms = keys.read()
        keff = oracle.reconstruct(_olayout(oracle, p), oracle.unpack(packed.reshape(T, -1), 128, p.nibbleDims),
                                  norms.view(np.float16).reshape(T, -1).astype(np.float32))
        for causal in (False, True):
            pos = np.array([0, 2047, 4095])
            out = att.attend(q, pos, causal)
            ins = att.inspect()
            rl, rp, ro = oracle.attention(q, keff, v, pos, causal)
            _check(out, ro.astype(np.float64), f"output causal={causal}")
            fin = np.isfinite(rl)
            assert np.array_equal(np.isneginf(ins["logits"]), np.isneginf(rl))
            np.testing.assert_allclose(ins["logits"][fin], rl[fin], atol=1e-4, rtol=2e-5)
            np.testing.assert_allclose(ins["probabilities"], rp, atol=1e-5, rtol=1e-4)
            if causal:
                np.testing.assert_array_equal(out[0], v[0])
    finally:
        att.destroy()
        values.destroy()
        keys.destroy()


def test_graph_replays_match_eager(device, oracle):
    """The decode captured in a HIP graph: every replay, with eager work between
    replays, equals the eager result (the split counters reset in-kernel, no
    memset nodes)."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    p = calibrate.layout_b(64)
    batch, hq, hkv, dim, T = 2, 14, 2, 64, 3000
    g = torch.Generator().manual_seed(21)
    k = torch.randn((batch, hkv, T, dim), generator=g).half().cuda()
    v = torch.randn((batch, hkv, T, dim), generator=g).half().cuda()
    q = torch.randn((batch, hq, dim), generator=g).cuda()
    tabs = [bgtq.Tables(device, p) for _ in range(hkv)]
    packed = torch.zeros((batch, hkv, T * p.rowBytes + 64), dtype=torch.uint8, device="cuda")
    norms = torch.zeros((batch, hkv, T * p.normStride + 32), dtype=torch.int16, device="cuda")
    batched.bind_torch_stream(device)
    batched.encode(device, [dict(tables=tabs[h], src=k[b, h], src_row_stride=dim, rows=T, packed=packed[b, h],
                                 norms=norms[b, h]) for b in range(batch) for h in range(hkv)], "f16")
    out = torch.empty((batch, hq, dim), device="cuda")
    lengths = torch.tensor([T, T - 123], dtype=torch.int32, device="cuda")
    args = dict(batch=batch, q_heads=hq, kv_heads=hkv, dim=dim, q=q, out=out, lengths=lengths, max_length=T, v=v,
                v_seq_stride=v.stride(0), v_head_stride=v.stride(1), tables=tabs, packed=packed,
                packed_seq_stride=packed.stride(0), packed_head_stride=packed.stride(1), norms=norms,
                norms_seq_stride=norms.stride(0), norms_head_stride=norms.stride(1), splits=5)
    ws = torch.zeros(batched.workspace_bytes(batched.decode_desc(**args)), dtype=torch.uint8, device="cuda")
    desc = batched.decode_desc(workspace=ws, **args)
    batched.decode(device, desc)
    torch.cuda.synchronize()
    eager = out.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        batched.bind_torch_stream(device)
        batched.decode(device, desc)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        batched.bind_torch_stream(device)
        batched.decode(device, desc)
    batched.bind_torch_stream(device)
    for rep in range(4):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {rep} differs from the eager result"
        batched.decode(device, desc)  # eager work between replays
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    for t in tabs:
        t.destroy()


def test_batch_beyond_grid_refused(device):
    """The fused kernel's grid carries the sequence in its third dimension (at most 65535): a larger batch
    is refused before any launch."""
    import torch
    import bgtq
    from bgtq import batched
    z = torch.zeros(16, device="cuda")
    args = dict(batch=65536, q_heads=2, kv_heads=1, dim=64, q=z, out=z, lengths=z, max_length=32, v=z, v_dtype="f16",
                v_seq_stride=0, v_head_stride=0, k_f16=z, k_seq_stride=0, k_head_stride=0, splits=1)
    with pytest.raises(bgtq.UnsupportedError, match="65535 sequences"):
        batched.workspace_bytes(batched.decode_desc(**args))


@pytest.mark.parametrize("key_format,layout,dim,hq,hkv,lengths", [
    ("packed", "B", 64, 14, 2, [1, 31, 33, 1000]), ("packed", "A", 64, 3, 1, [700, 129]),
    ("packed", "B", 128, 16, 4, [257, 64]), ("packed", "A", 128, 2, 2, [1, 500]),
    ("fp16", None, 64, 5, 1, [127, 128, 300]), ("fp16", None, 128, 8, 8, [65]),
])
def test_fp32_values_batched(device, oracle, key_format, layout, dim, hq, hkv, lengths):
    """bgtq_decode over FP32 V (its PV products on the FP32 matrix cores): values of ordinary size and, in
    one dimension, near the largest FP32, whose products with the probabilities must not overflow on the
    way. The rows past a sequence's length are NaN (never read into the result)."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    batched.bind_torch_stream(device)
    print("fp32 V batched", key_format, layout, dim, lengths, flush=True)
    g = torch.Generator().manual_seed(3)
    B, cap, G = len(lengths), max(lengths) + 9, hq // hkv
    k = (torch.randn((B, hkv, cap, dim), generator=g) * 0.8).half()
    v = torch.randn((B, hkv, cap, dim), generator=g)
    v[..., 5] *= 2.0e37
    q = torch.randn((B, hq, dim), generator=g)
    for b, n in enumerate(lengths):
        v[b, :, n:] = float("nan")
    kd, vd, qd = k.cuda(), v.cuda(), q.cuda()
    lens = torch.tensor(lengths, dtype=torch.int32).cuda()
    out = torch.empty((B, hq, dim), device="cuda")
    tabs = []
    if key_format == "packed":
        p = calibrate.layout_b(dim) if layout == "B" else calibrate.layout_a(dim)
        tabs = [bgtq.Tables(device, p) for _ in range(hkv)]
        packed = torch.zeros((B, hkv, (cap * p.rowBytes + 79) // 16 * 16), dtype=torch.uint8, device="cuda")
        norms = torch.zeros((B, hkv, (cap * p.normStride + 39) // 8 * 8), dtype=torch.int16, device="cuda")
        batched.encode(device, [dict(tables=tabs[h], src=kd[b, h], src_row_stride=dim, rows=cap, packed=packed[b, h],
                                     norms=norms[b, h]) for b in range(B) for h in range(hkv)], "f16")
        kw = dict(tables=tabs, packed=packed, packed_seq_stride=packed.stride(0), packed_head_stride=packed.stride(1),
                  norms=norms, norms_seq_stride=norms.stride(0), norms_head_stride=norms.stride(1))
    else:
        kw = dict(k_f16=kd, k_seq_stride=kd.stride(0), k_head_stride=kd.stride(1))
    args = dict(batch=B, q_heads=hq, kv_heads=hkv, dim=dim, q=qd, out=out, lengths=lens, max_length=max(lengths), v=vd,
                v_dtype="f32", v_seq_stride=vd.stride(0), v_head_stride=vd.stride(1), **kw)
    try:
        for splits in (0, 1, 3):
            ws = torch.zeros(batched.workspace_bytes(batched.decode_desc(splits=splits, **args)), dtype=torch.uint8,
                             device="cuda")
            out.fill_(float("nan"))
            batched.decode(device, batched.decode_desc(splits=splits, workspace=ws, **args))
            torch.cuda.synchronize()
            got = out.cpu().numpy()
            for b, T in enumerate(lengths):
                for h in range(hkv):
                    if key_format == "packed":
                        pk = packed[b, h, :T * p.rowBytes].cpu().numpy().reshape(T, p.rowBytes)
                        nm = norms[b, h, :T * p.normStride].cpu().numpy().view(np.float16).reshape(T, p.normStride)
                        keff = oracle.reconstruct(_olayout(oracle, p), oracle.unpack(pk, dim, p.nibbleDims),
                                                  nm.astype(np.float32))
                    else:
                        keff = k[b, h, :T].float().numpy()
                    vv = v[b, h, :T].numpy()
                    _, _, ref = oracle.attention(q[b, h * G:(h + 1) * G].numpy(), keff, vv, np.full(G, T - 1), False)
                    # The usual bar in units of each dimension's largest value (the sums' terms).
                    err = np.abs(got[b, h * G:(h + 1) * G].astype(np.float64) - ref)
                    big = np.maximum(1.0, np.abs(vv.astype(np.float64)).max(0))
                    lim = ATOL * big + RTOL * np.abs(ref.astype(np.float64))
                    assert np.all(err <= lim), f"splits {splits} b{b} kv{h}: worst ratio {(err / lim).max():.2f}"
    finally:
        for t in tabs:
            t.destroy()


@pytest.mark.parametrize("layout,dim,hq,hkv", [("A", 64, 9, 3), ("A", 64, 2, 1), ("B", 64, 14, 2), ("A", 128, 4, 2),
                                              ("B", 128, 8, 2)])
def test_fp32_values_keep_fp32_logits(device, oracle, layout, dim, hq, hkv):
    """bgtq_decode over FP32 V with logits of up to about 80 (the output's error then is the logits'): about
    as far from 64 bits as the same attention in plain FP32 on the CPU (query rotation, QK with the
    centroids, scales, softmax and PV). The bound is 1.35 times that error: the sums here are chains, the
    CPU's are blocked (FP32 chains measured 0.9 to 1.3 times it, 22-bit operands up to 1.9 times)."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    batched.bind_torch_stream(device)
    p = calibrate.layout_b(dim) if layout == "B" else calibrate.layout_a(dim)
    g = torch.Generator().manual_seed(dim + hq)
    B, T, G = 24, 1500, hq // hkv
    k = torch.randn((B, hkv, T, dim), generator=g).half()
    v = torch.randn((B, hkv, T, dim), generator=g).cuda()
    q = (torch.randn((B, hq, dim), generator=g) * 15).cuda()
    tables = bgtq.Tables(device, p)
    try:
        packed = torch.zeros((B, hkv, (T * p.rowBytes + 79) // 16 * 16), dtype=torch.uint8, device="cuda")
        norms = torch.zeros((B, hkv, (T * p.normStride + 39) // 8 * 8), dtype=torch.int16, device="cuda")
        kd = k.cuda()
        batched.encode(device, [dict(tables=tables, src=kd[b, h], src_row_stride=dim, rows=T, packed=packed[b, h],
                                     norms=norms[b, h]) for b in range(B) for h in range(hkv)], "f16")
        out = torch.empty((B, hq, dim), device="cuda")
        args = dict(batch=B, q_heads=hq, kv_heads=hkv, dim=dim, q=q, out=out, max_length=T, v=v, v_dtype="f32",
                    lengths=torch.full((B,), T, dtype=torch.int32, device="cuda"), v_seq_stride=v.stride(0),
                    v_head_stride=v.stride(1), tables=[tables] * hkv, packed=packed,
                    packed_seq_stride=packed.stride(0), packed_head_stride=packed.stride(1), norms=norms,
                    norms_seq_stride=norms.stride(0), norms_head_stride=norms.stride(1))
        ws = torch.zeros(batched.workspace_bytes(batched.decode_desc(**args)), dtype=torch.uint8, device="cuda")
        batched.decode(device, batched.decode_desc(workspace=ws, **args))
        torch.cuda.synchronize()
    finally:
        tables.destroy()
    perm, group_of = torch.tensor(np.asarray(p.permutation).astype(np.int64)), np.asarray(p.groupOf)
    cent = torch.tensor(np.asarray(p.centroids, np.float32).reshape(dim, -1))
    rot = torch.tensor(np.asarray(p.rotation, np.float32).reshape(dim, dim))
    refs = {torch.float32: [], torch.float64: []}
    largest = 0.0
    for b in range(B):
        for h in range(hkv):
            pk = packed[b, h, :T * p.rowBytes].cpu().numpy().reshape(T, p.rowBytes)
            codes = torch.tensor(oracle.unpack(pk, dim, p.nibbleDims).astype(np.int64))
            c32 = cent[torch.arange(dim)[None], codes]
            s32 = norms[b, h, :T * p.normStride].cpu().view(torch.float16).view(T, p.normStride)
            for dt, got in refs.items():
                qr = (q[b, h * G:(h + 1) * G].cpu().to(dt)[:, perm] @ rot.to(dt).t()) * torch.tensor(dim ** -0.5, dtype=dt)
                lg = torch.zeros((G, T), dtype=dt)
                for i in range(p.groups):
                    own = torch.tensor(np.nonzero(group_of == i)[0])
                    lg += (qr[:, own] @ c32.to(dt)[:, own].t()) * s32[:, i].to(dt)
                largest = max(largest, lg.abs().max().item())
                got.append(torch.softmax(lg, 1) @ v[b, h].cpu().to(dt))
    assert 40 < largest < 150
    ref = torch.cat(refs[torch.float64]).view(B, hq, dim)
    plain = (torch.cat(refs[torch.float32]).view(B, hq, dim).double() - ref).norm() / ref.norm()
    err = (out.cpu().double() - ref).norm() / ref.norm()
    print(f"fp32 logits {layout} d{dim}: error {err:.2e}, plain FP32 {plain:.2e}, logits to {largest:.0f}", flush=True)
    assert err <= 1.35 * plain, (err, plain)


def test_session_with_large_values_keeps_fp32_logits(device, oracle):
    """A session whose V reaches 65504 multiplies packed K in FP32 too: the bound above, over sixteen
    queries of three sessions, with logits of up to about 80."""
    import torch
    import bgtq
    from bgtq import calibrate
    p = calibrate.layout_a(64)
    rng = np.random.default_rng(8)
    T, errs, plains, norms2 = 1500, 0.0, 0.0, 0.0
    tables = bgtq.Tables(device, p)
    for _ in range(3):
        keys, values = bgtq.PackedKeys(device, tables, T), bgtq.Values(device, 64, T)
        session = bgtq.OptimizedAttention.create(device, keys, values, 16, materialize=False)
        try:
            keys.append(rng.standard_normal((T, 64)).astype(np.float16).view(np.uint16))
            v = (rng.standard_normal((T, 64)) * 1e5).astype(np.float32)
            values.append(v[:700])
            values.append(v[700:])
            q = (rng.standard_normal((16, 64)) * 15).astype(np.float32)
            out = torch.tensor(session.attend(q, np.zeros(16, np.uint32), False)).double()
            packed, norms = keys.read()
        finally:
            session.destroy()
            values.destroy()
            keys.destroy()
        codes = torch.tensor(oracle.unpack(packed[:T * p.rowBytes].reshape(T, -1), 64, p.nibbleDims).astype(np.int64))
        c = torch.tensor(np.asarray(p.centroids, np.float32).reshape(64, -1))[torch.arange(64)[None], codes]
        scale = torch.tensor(norms[:T * p.normStride].reshape(T, -1).view(np.float16).astype(np.float32))
        perm, rot = np.asarray(p.permutation), torch.tensor(np.asarray(p.rotation, np.float32).reshape(64, 64))
        outs = []
        for dt in (torch.float32, torch.float64):
            qr = (torch.tensor(q[:, perm]).to(dt) @ rot.to(dt).t()) * 0.125
            lg = torch.zeros((16, T), dtype=dt)
            for i in range(p.groups):
                own = torch.tensor(np.nonzero(np.asarray(p.groupOf) == i)[0])
                lg += (qr[:, own] @ c.to(dt)[:, own].t()) * scale[:, i].to(dt)
            outs.append((torch.softmax(lg, 1) @ torch.tensor(v).to(dt)).double())
        errs += float(((out - outs[1]) ** 2).sum())
        plains += float(((outs[0] - outs[1]) ** 2).sum())
        norms2 += float((outs[1] ** 2).sum())
    tables.destroy()
    print(f"large V session: error {(errs / norms2) ** 0.5:.2e}, plain FP32 {(plains / norms2) ** 0.5:.2e}", flush=True)
    assert errs <= 1.35 ** 2 * plains


@pytest.mark.parametrize("batch,hkv,ctx,fewer", [
    (150, 2, 3000, 2),  # 300 units: three splits where the rounded-up count is two
    (150, 2, 3000, 0),
    (257, 2, 200, 0),   # 514 units, just past the workgroup slots: one split
    (32, 8, 129, 0),    # 256 units, two splits of which the second holds one token
    (21, 3, 1500, 0),   # 63 units: eight splits, one workgroup per slot at most
])
def test_default_splits_by_rounds(device, batch, hkv, ctx, fewer):
    """The library's split choice at the edges of its rule, and a workspace sized for `fewer` splits
    (the call then takes those), against float64 attention."""
    import torch
    from bgtq import batched
    batched.bind_torch_stream(device)
    G, dim = 2, 64
    g = torch.Generator().manual_seed(batch)
    k = torch.randn((hkv, ctx, dim), generator=g).half()  # every sequence reads the same rows (stride 0)
    v = torch.randn((hkv, ctx, dim), generator=g).half()
    q = torch.randn((batch, hkv * G, dim), generator=g)
    lengths = [ctx if b % 50 == 0 else 1 + (37 * b) % min(ctx, 300) for b in range(batch)]
    out = torch.full((batch, hkv * G, dim), float("nan"), device="cuda")
    kd, vd = k.cuda(), v.cuda()
    kw = dict(batch=batch, q_heads=hkv * G, kv_heads=hkv, dim=dim, q=q.cuda(), out=out,
              lengths=torch.tensor(lengths, dtype=torch.int32).cuda(), max_length=ctx, v=vd, v_seq_stride=0,
              v_head_stride=ctx * dim, k_f16=kd, k_seq_stride=0, k_head_stride=ctx * dim)
    need = batched.workspace_bytes(batched.decode_desc(**kw))
    if fewer:
        small = batched.workspace_bytes(batched.decode_desc(splits=fewer, **kw))
        assert small < need
        need = small
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    print("default splits", batch, hkv, ctx, fewer, flush=True)
    for _ in range(2):
        batched.decode(device, batched.decode_desc(workspace=ws, **kw))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    for b in range(batch):
        n = lengths[b]
        for h in range(hkv):
            s = q[b, h * G:(h + 1) * G].double() @ k[h, :n].double().t() / dim ** 0.5
            _check(got[b, h * G:(h + 1) * G], (torch.softmax(s, 1) @ v[h, :n].double()).numpy(), f"b{b} kv{h} T={n}")
