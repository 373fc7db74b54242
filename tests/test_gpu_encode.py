"""K encode on the GPU: bit-exact against the reference goldens and the oracle.

Mirrors the checks of the reference's tests/test_mixed.py:38-64 (exact
packed bytes and scale bits) and tests/webgpu/optimized-test.ts:23-27 (an odd
append boundary, packed/norm buffers read back raw), through the C ABI.
"""
import json

import numpy as np
import pytest

from conftest import REF

pytestmark = pytest.mark.gpu


def _params(m, a):
    import bgtq
    return bgtq.BlockGTQParameters.from_mixed_fixture(m, a)


def _olayout(oracle, p):
    return oracle.Layout(dim=p.dim, groups=p.groups, row_bytes=p.rowBytes, norm_stride=p.normStride,
                         nibble_dims=p.nibbleDims, max_centroids=p.maxCentroids, perm=p.permutation,
                         group_of=p.groupOf, pos_to_cb=p.positionToCodebook, code_lut=p.codeLut,
                         rotation=p.rotation, centroids=p.centroids, offsets=p.offsets, inv_scales=p.inverseScales)


def test_mixed_fixture_rows_exact(device, mixed_cases):
    import bgtq
    for name, m, a in mixed_cases:
        print("case", name, flush=True)
        keys = bgtq.PackedKeys.create(device, _params(m, a), m["capacity"])
        try:
            x = a["original"].astype(np.float16).view(np.uint16)
            assert np.array_equal(x.view(np.float16).astype(np.float32), a["original"])
            keys.append(x[:2])
            keys.append(x[2:])
            packed, norms = keys.read()
            np.testing.assert_array_equal(packed, a["cache_packed"].reshape(-1), err_msg=name)
            np.testing.assert_array_equal(norms, a["cache_norms"].view(np.uint16).reshape(-1), err_msg=name)
            assert keys.length == m["rows"]
        finally:
            keys.destroy()


def test_attention_fixture_rows_exact(device, attention_cases):
    import bgtq
    for name, m, a, lm, la in attention_cases:
        print("case", name, flush=True)
        keys = bgtq.PackedKeys.create(device, _params(lm, la), m["context_length"])
        try:
            k = a["k"].view(np.uint16)
            keys.append(k[:3])  # odd row boundary shares packed words with the next append
            keys.append(k[3:])
            packed, norms = keys.read()
            np.testing.assert_array_equal(packed.reshape(a["packed_k"].shape), a["packed_k"], err_msg=name)
            np.testing.assert_array_equal(norms.reshape(a["norms"].shape), a["norms"].view(np.uint16), err_msg=name)
        finally:
            keys.destroy()


def _random_half_rows(rng, rows, dim):
    """FP16 K rows with mixed magnitudes: normal, tiny, subnormal, large, zeros, duplicates."""
    x = rng.standard_normal((rows, dim)).astype(np.float32)
    scale = np.exp(rng.uniform(-12, 8, size=(rows, 1))).astype(np.float32)
    x = (x * scale).clip(-60000, 60000)
    x[rng.random(rows) < 0.02] = 0.0
    x[rng.random((rows, dim)) < 0.01] = 0.0
    sub = rng.random(rows) < 0.01
    x[sub] = rng.integers(-1023, 1024, size=(int(sub.sum()), dim)).astype(np.float32) * 2.0 ** -24
    h = x.astype(np.float16)
    return h.view(np.uint16)


def _layouts(oracle):
    from bgtq import BlockGTQParameters
    out = []
    for name in ("low_d16", "mixed_d32", "mixed_d64", "low_d128", "mixed_d128", "awkward_all_widths", "only_high"):
        m, a = oracle.read_fixture(REF / "mixed" / f"{name}.json")
        out.append((name, BlockGTQParameters.from_mixed_fixture(m, a)))
    m, a = oracle.read_fixture(REF / "model" / "calibration.json")
    for i in (0, 1, 17, 89):
        out.append((f"smollm2_h{i}", BlockGTQParameters.from_serialized(a[f"h{i}_config"], a[f"h{i}_table"])))
    return out


def test_random_rows_bit_exact_vs_oracle(device, oracle):
    import bgtq
    rng = np.random.default_rng(2024)
    for name, p in _layouts(oracle):
        print("layout", name, flush=True)
        rows = 6000
        k = _random_half_rows(rng, rows, p.dim)
        ol = _olayout(oracle, p)
        ref_packed, ref_norms = oracle.encode_pack(ol, k)
        keys = bgtq.PackedKeys.create(device, p, rows + 5)
        try:
            cuts = [0, 1, 130, 257, 3000, rows]  # ragged appends
            for a, b in zip(cuts[:-1], cuts[1:]):
                keys.append(k[a:b])
            packed, norms = keys.read()
            packed = packed[: rows * p.rowBytes].reshape(rows, p.rowBytes)
            norms = norms[: rows * p.normStride].reshape(rows, p.normStride)
            bad = np.nonzero(np.any(packed != ref_packed, axis=1) | np.any(norms != ref_norms, axis=1))[0]
            assert bad.size == 0, f"{name}: {bad.size} rows differ, first {bad[:5]}"
        finally:
            keys.destroy()


def test_batched_encode_fp32_source_rounds_to_half(device, oracle):
    """Model path: FP32 post-RoPE rows [rows, kv_heads, dim], rounded to FP16 first (src/model/codec.wgsl:14)."""
    import torch
    import bgtq
    from bgtq import batched
    p = _layouts(oracle)[9][1]  # a real SmolLM2 head, d = 64
    tables = bgtq.Tables(device, p)
    rng = np.random.default_rng(7)
    rows, kvh = 1000, 3
    kr = (rng.standard_normal((rows, kvh, 64)) * 1.7).astype(np.float32)
    src = torch.from_numpy(kr).cuda()
    packed = torch.zeros((kvh, rows + 4, p.rowBytes), dtype=torch.uint8, device="cuda")
    norms = torch.zeros((kvh, rows + 4, p.normStride), dtype=torch.int16, device="cuda")
    jobs = [dict(tables=tables, src=src[:, h], src_row_stride=kvh * 64, rows=rows, packed=packed[h],
                 norms=norms[h], dst_row0=2) for h in range(kvh)]
    batched.encode(device, jobs, "f32")
    device.synchronize()
    ol = _olayout(oracle, p)
    for h in range(kvh):
        ref_p, ref_n = oracle.encode_pack(ol, kr[:, h].astype(np.float16).view(np.uint16))
        got_p = packed[h].cpu().numpy()
        got_n = norms[h].cpu().numpy().view(np.uint16)
        np.testing.assert_array_equal(got_p[2:2 + rows], ref_p)
        np.testing.assert_array_equal(got_n[2:2 + rows], ref_n)
        assert not got_p[:2].any() and not got_p[2 + rows:].any()
    tables.destroy()


def test_append_contracts(device, attention_cases):
    """appendCount and PackedKeys constructor rejections; failed calls leave state unchanged."""
    import bgtq
    name, m, a, lm, la = attention_cases[0]
    p = _params(lm, la)
    keys = bgtq.PackedKeys.create(device, p, 3)
    try:
        k = a["k"].view(np.uint16)
        with pytest.raises(bgtq.RangeError, match="whole nonempty rows"):
            keys.append(k[0, :5])
        with pytest.raises(bgtq.RangeError, match="whole nonempty rows"):
            keys.append(np.zeros(0, np.uint16))
        bad = k[:1].copy()
        bad[0, 3] = 0x7C00
        with pytest.raises(bgtq.RangeError, match="Finite FP16 K required"):
            keys.append(bad)
        with pytest.raises(bgtq.StateError, match="not ready"):
            keys.ready()
        keys.append(k[:3])
        with pytest.raises(bgtq.RangeError, match="K capacity exceeded"):
            keys.append(k[3:4])
        assert keys.length == 3
        keys.ready()
    finally:
        keys.destroy()
    changed = _params(lm, la)
    changed.rotation = changed.rotation.copy()
    grp = np.asarray(changed.groupOf)
    other = int(np.nonzero(grp != grp[0])[0][0])
    changed.rotation.reshape(p.dim, p.dim)[other, 0] = 0.01
    with pytest.raises(bgtq.StateError, match="Off-group transform is nonzero"):
        bgtq.PackedKeys.create(device, changed, 3)


def test_bulk_encode_bit_exact(device, oracle):
    """From 16384 rows a call leaves the wave-per-row encoder: d=16 takes the thread-per-row one, the d=64
    and d=128 layouts here the tile encoder through the device job table."""
    import torch
    import bgtq
    from bgtq import batched
    rng = np.random.default_rng(99)
    layouts = _layouts(oracle)
    for name, p in [layouts[i] for i in (0, 3, 9)]:
        print("bulk layout", name, flush=True)
        rows = 20000
        k = _random_half_rows(rng, rows, p.dim)
        ref_p, ref_n = oracle.encode_pack(_olayout(oracle, p), k)
        tables = bgtq.Tables(device, p)
        src = torch.from_numpy(k.view(np.int16)).cuda()
        packed = torch.zeros((rows, p.rowBytes), dtype=torch.uint8, device="cuda")
        norms = torch.zeros((rows, p.normStride), dtype=torch.int16, device="cuda")
        batched.encode(device, [dict(tables=tables, src=src, src_row_stride=p.dim, rows=rows, packed=packed,
                                     norms=norms)], "f16")
        device.synchronize()
        got_p, got_n = packed.cpu().numpy(), norms.cpu().numpy().view(np.uint16)
        bad = np.nonzero(np.any(got_p != ref_p, axis=1) | np.any(got_n != ref_n, axis=1))[0]
        assert bad.size == 0, f"{name}: {bad.size} rows differ, first {bad[:5]}"
        tables.destroy()


def test_bulk_layout_b_encoder_bit_exact(device, oracle):
    """Layout B tables (two equal groups, nibbles first), FP16 and FP32 sources, interleaved heads (row
    stride above dim), an offset destination. d=64: 270,000 rows, where FP16 sources take the bulk encoder
    with the layout's structure compiled in and FP32 sources the tile encoder, in a call that also carries
    a job of another layout kind. d=128: the tile encoder."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    rng = np.random.default_rng(123)
    other = _layouts(oracle)[2][1]  # mixed_d64: a launch of its own in the same call
    for dim in (64, 128):
        p = calibrate.layout_b(dim)
        print("bulk layout B", dim, flush=True)
        rows, heads, row0 = (90000 if dim == 64 else 20000), 3, 5
        k = _random_half_rows(rng, rows * heads, dim).reshape(rows, heads, dim)
        tables = bgtq.Tables(device, p)
        t_other = bgtq.Tables(device, other) if dim == 64 else None
        try:
            for src_kind in ("f16", "f32"):
                if src_kind == "f16":
                    src = torch.from_numpy(k.view(np.int16)).cuda()
                else:
                    src = torch.from_numpy(k.view(np.float16).astype(np.float32)).cuda()
                packed = torch.zeros((heads, row0 + rows, p.rowBytes), dtype=torch.uint8, device="cuda")
                norms = torch.zeros((heads, row0 + rows, p.normStride), dtype=torch.int16, device="cuda")
                jobs = [dict(tables=tables, src=src[:, h], src_row_stride=heads * dim, rows=rows, packed=packed[h],
                             norms=norms[h], dst_row0=row0) for h in range(heads)]
                if t_other is not None:
                    po = torch.zeros((rows, other.rowBytes), dtype=torch.uint8, device="cuda")
                    no = torch.zeros((rows, other.normStride), dtype=torch.int16, device="cuda")
                    jobs.append(dict(tables=t_other, src=src[:, 0], src_row_stride=heads * dim, rows=rows, packed=po,
                                     norms=no))
                batched.encode(device, jobs, src_kind)
                device.synchronize()
                for h in range(heads):
                    ref_p, ref_n = oracle.encode_pack(_olayout(oracle, p), np.ascontiguousarray(k[:, h]))
                    got_p = packed[h].cpu().numpy()
                    got_n = norms[h].cpu().numpy().view(np.uint16)
                    assert not got_p[:row0].any() and not got_n[:row0].any(), "rows before dst_row0 written"
                    bad = np.nonzero(np.any(got_p[row0:] != ref_p, axis=1) | np.any(got_n[row0:] != ref_n, axis=1))[0]
                    assert bad.size == 0, f"d={dim} {src_kind} head {h}: {bad.size} rows differ, first {bad[:5]}"
                if t_other is not None:
                    ref_p, ref_n = oracle.encode_pack(_olayout(oracle, other), np.ascontiguousarray(k[:, 0]))
                    assert np.array_equal(po.cpu().numpy(), ref_p)
                    assert np.array_equal(no.cpu().numpy().view(np.uint16), ref_n)
        finally:
            tables.destroy()
            if t_other is not None:
                t_other.destroy()


@pytest.mark.parametrize("dim", [64, 128])
def test_generic_encoder_bit_exact(device, oracle, dim):
    """A group boundary at an odd position is for neither the tile encoder nor the one with layout B's
    structure: from 16384 rows a call takes the generic thread-per-row encoder. Two jobs, one of them
    unaligned with an odd stride, FP16 and FP32, offset destinations with guard rows on both sides."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    rng = np.random.default_rng(64 + dim)
    p, cut = calibrate.layout_b(dim), dim // 2 - 1
    assert np.array_equal(p.groupOf, np.arange(dim) >= dim // 2)
    p.groupOf = (np.arange(dim) >= cut).astype(np.uint32)
    rot = np.zeros((dim, dim), np.float32)
    rot[:cut, :cut], rot[cut:, cut:] = calibrate.haar_rotation(cut, 1), calibrate.haar_rotation(dim - cut, 2)
    p.rotation = rot.reshape(-1)
    shapes = ((9001, dim + 1, 1, 3), (8000, dim, 0, 0))  # rows, stride, lead, row0
    ks = [_random_half_rows(rng, rows, dim) for rows, *_ in shapes]
    refs = [oracle.encode_pack(_olayout(oracle, p), k) for k in ks]
    tables = bgtq.Tables(device, p)
    try:
        for src_kind in ("f16", "f32"):
            jobs = []
            for (rows, stride, lead, row0), k in zip(shapes, ks):
                flat = np.zeros(lead + rows * stride, dtype=np.float16)
                flat[lead:].reshape(rows, stride)[:, :dim] = k.view(np.float16)
                src = torch.from_numpy(flat if src_kind == "f16" else flat.astype(np.float32)).cuda()
                n = row0 + rows + 2
                jobs.append(dict(tables=tables, src=src[lead:], src_row_stride=stride, rows=rows, dst_row0=row0,
                                 packed=torch.full((n, p.rowBytes), 0xA5, dtype=torch.uint8, device="cuda"),
                                 norms=torch.full((n, p.normStride), 0x5A5A, dtype=torch.int16, device="cuda")))
            batched.encode(device, jobs, src_kind)
            device.synchronize()
            for j, (rows, _, _, row0), (ref_p, ref_n) in zip(jobs, shapes, refs):
                got_p, got_n = j["packed"].cpu().numpy(), j["norms"].cpu().numpy().view(np.uint16)
                outside = np.r_[0:row0, row0 + rows:len(got_p)]
                assert np.all(got_p[outside] == 0xA5) and np.all(got_n[outside] == 0x5A5A), (src_kind, rows)
                assert np.array_equal(got_p[row0:row0 + rows], ref_p), (src_kind, rows)
                assert np.array_equal(got_n[row0:row0 + rows], ref_n), (src_kind, rows)
    finally:
        tables.destroy()


def test_bulk_encoder_unaligned_source(device, oracle):
    """The bulk encoder stages rows as 16-byte pieces when the source and its row stride allow it, else
    element-wise: 190,004 rows of layout B (one round of its workgroups) in three jobs, one starting past
    a 16-byte boundary with an odd stride, one with padded rows, one with only its start unaligned, FP16
    and FP32, partial last workgroups, offset destinations with guard rows on both sides."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    rng = np.random.default_rng(321)
    dim, guard = 64, 2
    p = calibrate.layout_b(dim)
    shapes = ((90001, dim + 1, 1, 3), (60000, dim + 8, 0, 0), (40003, dim, 3, 1))  # rows, stride, lead, row0
    ks = [_random_half_rows(rng, rows, dim) for rows, *_ in shapes]
    refs = [oracle.encode_pack(_olayout(oracle, p), np.ascontiguousarray(k)) for k in ks]
    tables = bgtq.Tables(device, p)
    try:
        for src_kind in ("f16", "f32"):
            jobs = []
            for (rows, stride, lead, row0), k in zip(shapes, ks):
                flat = np.zeros(lead + rows * stride, dtype=np.float16)
                flat[lead:].reshape(rows, stride)[:, :dim] = k.view(np.float16)
                src = torch.from_numpy(flat.view(np.int16) if src_kind == "f16" else flat.astype(np.float32)).cuda()
                n = row0 + rows + guard
                jobs.append(dict(tables=tables, src=src[lead:], src_row_stride=stride, rows=rows, dst_row0=row0,
                                 packed=torch.full((n, p.rowBytes), 0xA5, dtype=torch.uint8, device="cuda"),
                                 norms=torch.full((n, p.normStride), 0x5A5A, dtype=torch.int16, device="cuda")))
            batched.encode(device, jobs, src_kind)
            device.synchronize()
            for j, (rows, _, _, row0), (ref_p, ref_n) in zip(jobs, shapes, refs):
                got_p, got_n = j["packed"].cpu().numpy(), j["norms"].cpu().numpy().view(np.uint16)
                outside = np.r_[0:row0, row0 + rows:len(got_p)]
                assert np.all(got_p[outside] == 0xA5) and np.all(got_n[outside] == 0x5A5A), (src_kind, rows)
                assert np.array_equal(got_p[row0:row0 + rows], ref_p), (src_kind, rows)
                assert np.array_equal(got_n[row0:row0 + rows], ref_n), (src_kind, rows)
    finally:
        tables.destroy()


@pytest.mark.parametrize("src_kind", ["f16", "f32"])
@pytest.mark.parametrize("dim,layouts", [(64, ("B", "A", "mixed_d64", "smollm2_h0", "smollm2_h17", "smollm2_h89")),
                                         (128, ("B", "A", "mixed_d128", "low_d128"))])
def test_tile_encoder_bit_exact(device, oracle, dim, layouts, src_kind):
    """One launch of jobs above the wave encoder's row limit takes the tile encoder (16 rows per wave):
    layouts of one to six groups, row counts around whole tiles, jobs with and without rows, interleaved
    heads, unaligned sources with odd strides, destinations at odd bytes with guard rows on both sides."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    rng = np.random.default_rng(77 + dim)
    known = dict(_layouts(oracle), B=calibrate.layout_b(dim), A=calibrate.layout_a(dim))
    print("tile encoder", dim, src_kind, flush=True)
    jobs, checks, tabs = [], [], []
    try:
        for i, name in enumerate(layouts):
            p = known[name]
            tabs.append(bgtq.Tables(device, p))
            for j, rows in enumerate((1, 15, 16, 17, 63, 1039, 3001) if i else (0, 5, 32, 4100)):
                stride = dim + (0, 8, 1)[j % 3]
                lead = (j % 2) * (1 if src_kind == "f32" else 3)  # elements before the first row
                row0, guard = (3, 0, 1, 2)[j % 4], 2
                k = _random_half_rows(rng, rows, dim)
                flat = np.zeros(lead + max(1, rows) * stride, dtype=np.float16)
                flat[lead:].reshape(-1, stride)[:rows, :dim] = k.view(np.float16)
                src = torch.from_numpy(flat if src_kind == "f16" else flat.astype(np.float32)).cuda()
                packed = torch.full((row0 + rows + guard, p.rowBytes), 0xA5, dtype=torch.uint8, device="cuda")
                norms = torch.full((row0 + rows + guard, p.normStride), 0x5A5A, dtype=torch.int16, device="cuda")
                jobs.append(dict(tables=tabs[-1], src=src[lead:], src_row_stride=stride, rows=rows, packed=packed,
                                 norms=norms, dst_row0=row0))
                checks.append((name, p, rows, row0, k, packed, norms))
        batched.encode(device, jobs, src_kind)
        device.synchronize()
        for name, p, rows, row0, k, packed, norms in checks:
            got_p, got_n = packed.cpu().numpy(), norms.cpu().numpy().view(np.uint16)
            outside = np.r_[0:row0, row0 + rows:len(got_p)]
            assert np.all(got_p[outside] == 0xA5) and np.all(got_n[outside] == 0x5A5A), f"{name} {rows}: guard rows"
            if rows:
                ref_p, ref_n = oracle.encode_pack(_olayout(oracle, p), np.ascontiguousarray(k))
                bad = np.nonzero(np.any(got_p[row0:row0 + rows] != ref_p, axis=1)
                                 | np.any(got_n[row0:row0 + rows] != ref_n, axis=1))[0]
                assert bad.size == 0, f"{name} {rows} rows: {bad.size} differ, first {bad[:5]}"
    finally:
        for t in tabs:
            t.destroy()


def _tree_sum(v):
    """ATen's FP32 inner sum of one row (d 64 or 128): 8 lanes of four interleaved accumulators."""
    total = np.float32(0)
    for lane in range(8):
        a = [np.float32(0)] * 4
        for i, x in enumerate(v[lane::8]):
            a[i % 4] = np.float32(a[i % 4] + x)
        part = np.float32(np.float32(np.float32(a[0] + a[1]) + a[2]) + a[3])
        total = np.float32(total + part)
    return total


def _encode_nonfinite(oracle, p, k, whole_rows):
    """Packed rows and scales of FP16 rows that may hold infinities and NaNs. A group that holds one has
    the scale inf or NaN over its centroids, and a group whose FMA chain (the 8-wide blocks it touches,
    or the whole row) meets one has every code at bin 0; all else is as with zeros in their place."""
    x = k.view(np.float16)
    clean = np.where(np.isfinite(x), x, np.float16(0))
    ref_p, ref_n = oracle.encode_pack(_olayout(oracle, p), np.ascontiguousarray(clean).view(np.uint16))
    ref_p, ref_n = ref_p.copy(), ref_n.copy()
    perm, group_of = np.asarray(p.permutation), np.asarray(p.groupOf)
    bin0 = np.asarray(p.codeLut).reshape(-1, 256)[np.asarray(p.positionToCodebook), 0]
    cent = np.asarray(p.centroids, np.float32).reshape(p.dim, -1)
    for r in np.nonzero(~np.isfinite(x).all(axis=1))[0]:
        v, z = x[r, perm].astype(np.float32), clean[r, perm].astype(np.float32)
        bad = ~np.isfinite(v)
        nib = p.nibbleDims
        codes = np.r_[np.stack([ref_p[r, :nib // 2] & 15, ref_p[r, :nib // 2] >> 4], 1).ravel(),
                      ref_p[r, nib // 2:nib // 2 + p.dim - nib]]
        for g in range(p.groups):
            at = np.nonzero(group_of == g)[0]
            span = slice(None) if whole_rows else slice(at[0] // 8 * 8, (at[-1] + 8) // 8 * 8)
            if bad[span].any():
                codes[at] = bin0[at]
        for g in range(p.groups):
            own = group_of == g
            n = np.sqrt(np.float32(_tree_sum(np.where(own, z * z, np.float32(0))) + np.float32(1e-30)))
            raw = np.float32(_tree_sum(np.where(own, n, np.float32(0))) / np.float32(own.sum())) if p.groups > 1 else n
            if bad[own].any():
                raw = np.float32(np.nan if np.isnan(v[own]).any() else np.inf)
            c = cent[np.arange(p.dim), codes]
            s = np.sqrt(_tree_sum(np.where(own, c * c, np.float32(0))))
            ref_n[r, g] = np.float16(raw / max(s, np.float32(1e-10))).view(np.uint16)
        ref_p[r, :nib // 2] = codes[0:nib:2] | codes[1:nib:2] << 4
        ref_p[r, nib // 2:nib // 2 + p.dim - nib] = codes[nib:]
    return ref_p, ref_n


@pytest.mark.parametrize("dim,name", [(64, "B"), (64, "A"), (64, "mixed_d64"), (64, "smollm2_h0"), (64, "smollm2_h17"),
                                      (128, "B"), (128, "A"), (128, "mixed_d128")])
def test_nonfinite_rows_keep_to_their_groups(device, oracle, dim, name):
    """Infinities (an FP32 value above 65504 is one) and NaNs among the rows of a tile-encoder call: the
    other rows and the row's other groups are as without them, in calls below and from 16384 rows."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    p = dict(_layouts(oracle), B=calibrate.layout_b(dim), A=calibrate.layout_a(dim))[name]
    rng = np.random.default_rng(dim)
    tables = bgtq.Tables(device, p)
    try:
        for rows in (9001, 16400):
            k = _random_half_rows(rng, rows, dim)
            f = k.view(np.float16)
            for r in rng.choice(rows, 60, replace=False):
                for c in rng.choice(dim, rng.choice([1, 1, 2, dim // 3]), replace=False):
                    f[r, c] = rng.choice(np.array([np.inf, -np.inf, np.nan], np.float16))
            f[37, :] = np.inf
            ref_p, ref_n = _encode_nonfinite(oracle, p, k, rows < 16384)
            for src_kind in ("f16", "f32"):
                x = f.astype(np.float32)
                x = np.where(np.isinf(x), np.copysign(np.float32(70000), x), x)
                src = torch.from_numpy(f if src_kind == "f16" else x).cuda()
                packed = torch.zeros((rows, p.rowBytes), dtype=torch.uint8, device="cuda")
                norms = torch.zeros((rows, p.normStride), dtype=torch.int16, device="cuda")
                batched.encode(device, [dict(tables=tables, src=src, src_row_stride=dim, rows=rows, packed=packed,
                                             norms=norms)], src_kind)
                device.synchronize()
                got_p, got_n = packed.cpu().numpy(), norms.cpu().numpy().view(np.uint16)
                same = (got_n == ref_n) | (np.isnan(got_n.view(np.float16)) & np.isnan(ref_n.view(np.float16)))
                bad = np.nonzero(np.any(got_p != ref_p, axis=1) | ~same.all(axis=1))[0]
                assert bad.size == 0, f"{rows} rows {src_kind}: {bad.size} differ, first {bad[:5]}"
    finally:
        tables.destroy()


def test_bulk_layout_b_largest_calls(device, oracle):
    """Layout B at d=64 where the thread-per-row encoder's second round of workgroups is well filled: FP16
    and FP32 sources, a partial last workgroup."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    rng = np.random.default_rng(5)
    p, rows = calibrate.layout_b(64), 380077
    k = _random_half_rows(rng, rows, 64)
    ref_p, ref_n = oracle.encode_pack(_olayout(oracle, p), k)
    tables = bgtq.Tables(device, p)
    try:
        for src_kind in ("f16", "f32"):
            src = torch.from_numpy(k.view(np.float16) if src_kind == "f16" else
                                   k.view(np.float16).astype(np.float32)).cuda()
            packed = torch.zeros((rows, p.rowBytes), dtype=torch.uint8, device="cuda")
            norms = torch.zeros((rows, p.normStride), dtype=torch.int16, device="cuda")
            batched.encode(device, [dict(tables=tables, src=src, src_row_stride=64, rows=rows, packed=packed,
                                         norms=norms)], src_kind)
            device.synchronize()
            assert np.array_equal(packed.cpu().numpy(), ref_p), src_kind
            assert np.array_equal(norms.cpu().numpy().view(np.uint16), ref_n), src_kind
    finally:
        tables.destroy()


def test_calibration_load_encodes_every_head(device, oracle):
    """Calibration.load (src/model/calibration.ts:7-21) puts the 90 SmolLM2 heads on the device;
    each head's tables then encode its KV head's post-RoPE rows bit for bit as the oracle does
    with the same blob (the reference's tests/webgpu/model-codec-test.ts:13-21 on 3 rows per
    head; here 37 rows, FP32 model-path source)."""
    import torch
    import bgtq
    from bgtq import batched
    cal = bgtq.Calibration.load(device, REF / "model")
    try:
        assert len(cal.heads) == 90 and len(cal.allocations) == 90
        assert all(x["bytes"] > 0 for x in cal.allocations)
        m, a = oracle.read_fixture(REF / "model" / "calibration.json")
        rng = np.random.default_rng(90)
        rows, kvh = 37, 3
        kr = (rng.standard_normal((rows, kvh, 64)) * 2.3).astype(np.float32)
        src = torch.from_numpy(kr).cuda()
        outs, jobs = [], []
        for h, head in enumerate(cal.heads):
            p = bgtq.BlockGTQParameters.from_serialized(a[f"h{h}_config"], a[f"h{h}_table"])
            info = head.tables.info
            assert (info["dim"], info["groups"], info["row_bytes"], info["norm_stride"]) == \
                (64, p.groups, p.rowBytes, p.normStride) == (64, p.groups, head.row_bytes, head.norm_stride)
            packed = torch.zeros((rows, p.rowBytes), dtype=torch.uint8, device="cuda")
            norms = torch.zeros((rows, p.normStride), dtype=torch.int16, device="cuda")
            outs.append((p, packed, norms))
            jobs.append(dict(tables=head.tables, src=src[:, h % kvh], src_row_stride=kvh * 64, rows=rows,
                             packed=packed, norms=norms, dst_row0=0))
        batched.encode(device, jobs, "f32")
        device.synchronize()
        for h, (p, packed, norms) in enumerate(outs):
            ref_p, ref_n = oracle.encode_pack(_olayout(oracle, p), kr[:, h % kvh].astype(np.float16).view(np.uint16))
            np.testing.assert_array_equal(packed.cpu().numpy(), ref_p, err_msg=f"head {h}")
            np.testing.assert_array_equal(norms.cpu().numpy().view(np.uint16), ref_n, err_msg=f"head {h}")
    finally:
        cal.destroy()


def test_job_table_batches_and_stream_switch(device, oracle):
    """More jobs in one call than the context's device job table holds (4100 jobs of 4 rows: two table
    batches, each uploaded in chunks of 60), then, without waiting, a second call on another stream that
    rewrites the table: both calls give the oracle's bytes."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    rng = np.random.default_rng(321)
    p = calibrate.layout_b(64)
    n_a, rows_a = 4100, 4
    n_b, rows_b = 90, 200
    ka = _random_half_rows(rng, n_a * rows_a, 64)
    kb = _random_half_rows(rng, n_b * rows_b, 64)
    tables = bgtq.Tables(device, p)
    side_a, side_b = torch.cuda.Stream(), torch.cuda.Stream()
    try:
        bufs = []
        for k in (ka, kb):
            src = torch.from_numpy(k.view(np.int16)).cuda()
            packed = torch.zeros((k.shape[0], p.rowBytes), dtype=torch.uint8, device="cuda")
            norms = torch.zeros((k.shape[0], p.normStride), dtype=torch.int16, device="cuda")
            bufs.append((src, packed, norms))
        torch.cuda.synchronize()

        def jobs(buf, n, rows):
            src, packed, norms = buf
            return [dict(tables=tables, src=src[i * rows:], src_row_stride=64, rows=rows,
                         packed=packed[i * rows:], norms=norms[i * rows:]) for i in range(n)]

        device.set_stream(side_a.cuda_stream)
        batched.encode(device, jobs(bufs[0], n_a, rows_a), "f16")
        device.set_stream(side_b.cuda_stream)
        batched.encode(device, jobs(bufs[1], n_b, rows_b), "f16")
        torch.cuda.synchronize()
        for name, k, (_, packed, norms) in (("table batches", ka, bufs[0]), ("second stream", kb, bufs[1])):
            ref_p, ref_n = oracle.encode_pack(_olayout(oracle, p), k)
            got_p, got_n = packed.cpu().numpy(), norms.cpu().numpy().view(np.uint16)
            bad = np.nonzero(np.any(got_p != ref_p, axis=1) | np.any(got_n != ref_n, axis=1))[0]
            assert bad.size == 0, f"{name}: {bad.size} rows differ, first {bad[:5]}"
    finally:
        device.set_stream(None)
        torch.cuda.synchronize()
        tables.destroy()


@pytest.mark.parametrize("dim,rows,heads", [(64, 3333, 3), (64, 100, 130), (128, 2048, 5)])
def test_small_encode_shares_no_table(device, oracle, dim, rows, heads):
    """A call below 16384 rows carries its jobs in kernel arguments (more jobs than one launch holds,
    several launches): its captured graph replays on another stream while the same context encodes
    eagerly through the device job table, and both keep giving the oracle's bytes."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    rng = np.random.default_rng(11)
    p = calibrate.layout_a(dim)
    small, large = heads * rows, 17000
    assert small < 16384
    k, kl = _random_half_rows(rng, small, dim), _random_half_rows(rng, large, dim)
    tables = bgtq.Tables(device, p)
    side, main = torch.cuda.Stream(), torch.cuda.Stream()
    try:
        def buffers(x):
            return (torch.from_numpy(x.view(np.int16)).cuda(),
                    torch.zeros((len(x), p.rowBytes), dtype=torch.uint8, device="cuda"),
                    torch.zeros((len(x), p.normStride), dtype=torch.int16, device="cuda"))

        def jobs(b, n, r):
            return [dict(tables=tables, src=b[0][i * r:], src_row_stride=dim, rows=r, packed=b[1][i * r:],
                         norms=b[2][i * r:]) for i in range(n)]

        bs, bl = buffers(k), buffers(kl)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            device.set_stream(torch.cuda.current_stream().cuda_stream)
            batched.encode(device, jobs(bs, heads, rows), "f16")
        device.set_stream(main.cuda_stream)
        ref = [oracle.encode_pack(_olayout(oracle, p), x) for x in (k, kl)]
        for trial in range(6):
            print("replay", dim, heads, trial, flush=True)
            for t in (*bs[1:], *bl[1:]):
                t.zero_()
            torch.cuda.synchronize()
            for _ in range(4):
                with torch.cuda.stream(side):
                    graph.replay()
                batched.encode(device, jobs(bl, 17, large // 17), "f16")
            torch.cuda.synchronize()
            for (rp, rn), b in zip(ref, (bs, bl)):
                assert np.array_equal(b[1].cpu().numpy(), rp)
                assert np.array_equal(b[2].cpu().numpy().view(np.uint16), rn)
    finally:
        torch.cuda.synchronize()
        device.set_stream(None)
        tables.destroy()


@pytest.mark.parametrize("dim,lengths", [(64, [8001] + [1] * 40), (64, [20011] + [3] * 75 + [700]), (64, [9000] + [1] * 130),
                                         (128, [5003] + [17] * 9), (128, [16385] + [2] * 61)])
def test_one_long_job_among_short_ones(device, oracle, dim, lengths):
    """A long job beside many short ones is cut into parts (calls below and from 16384 rows): odd strides,
    odd destination rows, guard rows on both sides."""
    import torch
    import bgtq
    from bgtq import batched, calibrate
    rng = np.random.default_rng(len(lengths))
    names = ("smollm2_h0", "smollm2_h17", "mixed_d64") if dim == 64 else ("A", "mixed_d128")
    known = dict(_layouts(oracle), A=calibrate.layout_a(dim))
    tabs = [bgtq.Tables(device, known[n]) for n in names]
    try:
        for src_kind in ("f16", "f32"):
            jobs, checks = [], []
            for i, rows in enumerate(lengths):
                p, row0, stride = known[names[i % len(names)]], i % 4, dim + (1, 8, 0)[i % 3]
                k = _random_half_rows(rng, rows, dim)
                flat = np.zeros((rows, stride), np.float16)
                flat[:, :dim] = k.view(np.float16)
                src = torch.from_numpy(flat if src_kind == "f16" else flat.astype(np.float32)).cuda()
                packed = torch.full((row0 + rows + 2, p.rowBytes), 0xA5, dtype=torch.uint8, device="cuda")
                norms = torch.full((row0 + rows + 2, p.normStride), 0x5A5A, dtype=torch.int16, device="cuda")
                jobs.append(dict(tables=tabs[i % len(names)], src=src, src_row_stride=stride, rows=rows, packed=packed,
                                 norms=norms, dst_row0=row0))
                checks.append((p, row0, k, packed, norms))
            batched.encode(device, jobs, src_kind)
            device.synchronize()
            for i, (p, row0, k, packed, norms) in enumerate(checks):
                ref_p, ref_n = oracle.encode_pack(_olayout(oracle, p), k)
                got_p, got_n = packed.cpu().numpy(), norms.cpu().numpy().view(np.uint16)
                own = slice(row0, row0 + len(k))
                assert np.array_equal(got_p[own], ref_p) and np.array_equal(got_n[own], ref_n), f"job {i} {src_kind}"
                outside = np.r_[0:row0, row0 + len(k):len(got_p)]
                assert np.all(got_p[outside] == 0xA5) and np.all(got_n[outside] == 0x5A5A), f"job {i}: guard rows"
    finally:
        for t in tabs:
            t.destroy()


def test_concurrent_appends_near_capacity(device, oracle):
    """Two threads append at once near the end of a store's capacity (the Node addon runs appends off
    the JS thread). The store is claimed before the capacity check, as the reference refuses a second
    append while one is in flight (src/runtime/packed-keys.ts:40-49): each append either completes or
    is refused ("Concurrent K appends unsupported" while the other runs, "K capacity exceeded" after
    it committed), never both complete, the length counts the completed rows, and the committed rows
    are the oracle's encode of the base rows and the winning append."""
    import threading
    import bgtq
    from bgtq import calibrate
    p = calibrate.layout_b(64)
    ol = _olayout(oracle, p)
    rng = np.random.default_rng(77)
    cap, base_rows, add = 96, 80, 12
    outcomes = set()
    for trial in range(24):
        keys = bgtq.PackedKeys.create(device, p, cap)
        try:
            base = _random_half_rows(rng, base_rows, 64)
            keys.append(base)
            batches = [_random_half_rows(rng, add, 64) for _ in range(2)]
            results = [None, None]
            gate = threading.Barrier(2)

            def run(i):
                gate.wait()
                try:
                    keys.append(batches[i])
                    results[i] = "ok"
                except (bgtq.StateError, bgtq.RangeError) as e:
                    results[i] = str(e)

            threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
            for t in threads:
                t.start()
            for t in threads:
                t.join()
            assert results.count("ok") == 1, results
            for r in results:
                assert r in ("ok", "Concurrent K appends unsupported", "K capacity exceeded"), r
            outcomes.add(tuple(sorted(results)))
            winner = results.index("ok")
            assert keys.length == base_rows + add
            rows = base_rows + add
            ref_p, ref_n = oracle.encode_pack(ol, np.concatenate([base, batches[winner]]))
            packed, norms = keys.read()
            np.testing.assert_array_equal(packed[: rows * p.rowBytes].reshape(rows, -1), ref_p)
            np.testing.assert_array_equal(norms[: rows * p.normStride].reshape(rows, -1), ref_n)
            assert not packed[rows * p.rowBytes:].any(), "rows past the length were written"
            with pytest.raises(bgtq.RangeError, match="K capacity exceeded"):
                keys.append(batches[1 - winner])
        finally:
            keys.destroy()
    print("outcomes", sorted(outcomes), flush=True)
