"""GPU parity for shapes with no compiled kernel: any GQA group and any even head_dim up to
256 on the reference's dispatch surface (attention_op, rope_op, the fused layer step) and
the fp32 batched / ragged decode.  The reference's attention_op sends head_dim != 64 to
kernel_attn, which takes any group and head_dim (metal_backend.hpp:416-452,
kernel_attn.metal:7-60), and kernel_rope takes any head_dim (kernel_rope.metal:5-22).

Oracle: oracle/tmac_oracle.c (tmac_gguf.cpp:990-1016 RoPE, 1093-1128 attention with the
scale 1/sqrt(head_dim)).  Attention within 2e-5 + 1e-4 |ref|; RoPE and cache rows
bit-exact.  Entry points and cache types that keep head_dim 64 and the compiled groups
must refuse other shapes with TMAC_ERR_UNSUPPORTED."""
import numpy as np
import pytest

import oracle
import tmac_attn
from conftest import assert_close

pytestmark = pytest.mark.gpu

SHAPES = [(3, 1, 64), (6, 3, 64), (14, 2, 32), (14, 2, 128), (8, 8, 80), (12, 4, 96), (2, 1, 2), (5, 5, 256),
          (16, 2, 128), (9, 3, 66)]


@pytest.mark.parametrize("nh,nkv,hd", SHAPES)
@pytest.mark.parametrize("past_len", [0, 5, 255, 1000])
def test_attention_op_any_shape(ctx, nh, nkv, hd, past_len):
    n = past_len + 1
    k = oracle.normal(7000 + hd + past_len, (n, nkv * hd))
    v = oracle.normal(7001 + hd + past_len, (n, nkv * hd))
    q = oracle.normal(7002 + nh + past_len, nh * hd)
    dq, dk, dv, dout = ctx.upload(q), ctx.upload(k), ctx.upload(v), ctx.empty(nh * hd)
    ctx.attention_op(dq, dk, dv, dout, nh, nkv, hd, past_len)
    assert_close(dout.numpy(), oracle.attention(q, k, v, nh, nkv, hd, past_len),
                 f"attention_op heads {nh}/{nkv} head_dim {hd} past_len {past_len}")
    assert ctx.check_device_error() == 0


@pytest.mark.parametrize("hd", [2, 32, 66, 80, 128, 256])
def test_rope_any_head_dim_bit_exact(ctx, hd):
    for n_heads, pos in ((3, 0), (5, 17), (2, 4095), (7, 300000)):
        x = oracle.normal(7100 + hd + pos, n_heads * hd)
        d = ctx.upload(x)
        ctx.rope_op(d, n_heads, hd, pos, 1e6)
        np.testing.assert_array_equal(d.numpy(), oracle.rope_heads(x, n_heads, hd, pos, 1e6))
    rows, stride, n_heads = 9, 4 * hd + 8, 4
    x = oracle.normal(7150 + hd, (rows, stride))
    d = ctx.upload(x)
    ctx.rope_rows(d, rows, stride, n_heads, hd, 100, 1e4)
    got = d.numpy()
    for r in range(rows):
        np.testing.assert_array_equal(got[r, :n_heads * hd], oracle.rope_heads(x[r, :n_heads * hd], n_heads, hd,
                                                                              100 + r, 1e4))
    np.testing.assert_array_equal(got[:, n_heads * hd:], x[:, n_heads * hd:])
    assert ctx.check_device_error() == 0


@pytest.mark.parametrize("nh,nkv,hd", [(3, 1, 64), (14, 2, 128), (12, 4, 96), (9, 3, 66)])
def test_batched_and_ragged_any_shape(ctx, nh, nkv, hd):
    n_seq, n_pos = 5, 300
    k = oracle.normal(7200 + hd, (n_seq * n_pos, nkv * hd))
    v = oracle.normal(7201 + hd, (n_seq * n_pos, nkv * hd))
    q = oracle.normal(7202 + hd, (n_seq, nh * hd))
    offs = np.arange(n_seq, dtype=np.int64) * n_pos
    ref = oracle.attention_ragged(q, k, v, offs, np.full(n_seq, n_pos, np.int32), nh, nkv, hd, n_threads=8)
    dq, dk, dv, dout = ctx.upload(q), ctx.upload(k), ctx.upload(v), ctx.empty((n_seq, nh * hd))
    ctx.decode_batched(dq, dk, dv, dout, n_seq, nh, nkv, hd, n_pos, n_pos)
    assert_close(dout.numpy(), ref, f"batched {nh}/{nkv}/{hd}")
    lens = np.array([1, 0, 300, 77, 2999], np.int32)
    offs = np.concatenate([[0], np.cumsum(lens[:-1])]).astype(np.int64)
    kr = oracle.normal(7210 + hd, (int(lens.sum()), nkv * hd))
    vr = oracle.normal(7211 + hd, (int(lens.sum()), nkv * hd))
    nz = lens > 0
    ref = np.zeros((lens.size, nh * hd), np.float32)
    ref[nz] = oracle.attention_ragged(q[nz], kr, vr, offs[nz], lens[nz], nh, nkv, hd, n_threads=8)
    dk, dv, do, dl = ctx.upload(kr), ctx.upload(vr), ctx.upload(offs), ctx.upload(lens)
    ctx.decode_ragged(dq, dk, dv, do, dl, dout, lens.size, nh, nkv, hd, 3000)
    assert_close(dout.numpy(), ref, f"ragged {nh}/{nkv}/{hd}")
    ctx.decode_ragged(dq, dk, dv, do, dl, dout, lens.size, nh, nkv, hd, 1000)  # 2999 > max_len: NaN, bit 1
    assert np.all(np.isnan(dout.numpy()[4]))
    assert ctx.check_device_error() == tmac_attn.TMAC_ERR_DEVICE_FAULT
    assert ctx.query_split(4, 300, nh, nkv) == (300, 0)


@pytest.mark.parametrize("nh,nkv,hd", [(3, 1, 64), (14, 2, 128), (8, 8, 80), (9, 3, 66)])
def test_layer_step_any_shape(ctx, nh, nkv, hd):
    """Fused RoPE + cache write + attention, host and device positions, against the
    reference's sequence (tmac_gguf.cpp:1085-1128); cache rows bit-exact."""
    cap = 64
    kc = np.zeros((cap, nkv * hd), np.float32)
    vc = np.zeros((cap, nkv * hd), np.float32)
    dkc, dvc, dout = ctx.upload(kc), ctx.upload(vc), ctx.empty(nh * hd)
    pos_dev = ctx.upload(np.zeros(1, np.int32))
    ctx.rope_prepare(hd, 1e6, cap)
    for pos in range(40):
        q = oracle.normal(7300 + pos, nh * hd)
        kn = oracle.normal(7400 + pos, nkv * hd)
        vn = oracle.normal(7500 + pos, nkv * hd)
        dq, dkn, dvn = ctx.upload(q), ctx.upload(kn), ctx.upload(vn)
        if pos % 2:
            ctx.layer_attention(dq, dkn, dvn, dkc, dvc, dout, nh, nkv, hd, pos, cap, 1e6)
        else:
            pos_dev.copy_from(np.array([pos], np.int32))
            ctx.layer_attention_devpos(dq, dkn, dvn, dkc, dvc, dout, nh, nkv, hd, pos_dev, cap, 1e6)
        ref, _, _ = oracle.layer_step(q, kn, vn, kc, vc, nh, nkv, hd, pos, 1e6)
        assert_close(dout.numpy(), ref, f"layer {nh}/{nkv}/{hd} pos {pos}")
    np.testing.assert_array_equal(dkc.numpy(), kc)
    np.testing.assert_array_equal(dvc.numpy(), vc)
    assert ctx.check_device_error() == 0


@pytest.mark.parametrize("nh,nkv,hd", [(2, 1, 2), (14, 2, 32), (14, 2, 128)])
def test_layer_step_any_shape_counter_far_positions(ctx, nh, nkv, hd):
    """A device-side position counter read by the any-shape layer step and moved by
    tmac_pos_update (set, then advanced by one) to positions far past rows * hd / 64
    of a 4096-row RoPE table (127 for hd 2, 2047 for hd 32), up to the last row.  The
    counter first serves a head_dim-64 layer step (whose kernel keeps the counter's
    cached RoPE row), so the advances also refresh that cache from the head_dim-64
    table.  Both layer steps match the oracle (tmac_gguf.cpp:1085-1128) at every
    position, the cache rows bit-exact, and no device error is raised."""
    cap = 4096
    kc = oracle.normal(7600 + hd, (cap, nkv * hd))
    vc = oracle.normal(7601 + hd, (cap, nkv * hd))
    k64 = oracle.normal(7602, (cap, 128))
    v64 = oracle.normal(7603, (cap, 128))
    dkc, dvc, dout = ctx.upload(kc), ctx.upload(vc), ctx.empty(nh * hd)
    dk64, dv64, dout64 = ctx.upload(k64), ctx.upload(v64), ctx.empty(14 * 64)
    pos_dev = ctx.upload(np.zeros(1, np.int32))
    ctx.rope_prepare(hd, 1e6, cap)
    ctx.rope_prepare(64, 1e6, cap)
    s = ctx.stream()
    try:
        for i, (pos, how) in enumerate([(0, "set"), (126, "set"), (127, "add"), (128, "add"), (2046, "set"),
                                        (2047, "add"), (2048, "add"), (4094, "set"), (4095, "add")]):
            if how == "set":
                ctx.pos_update(pos_dev, pos, stream=s)
            else:
                ctx.pos_update(pos_dev, 1, add=True, stream=s)
            q64 = oracle.normal(7610 + i, 14 * 64)
            kn64, vn64 = oracle.normal(7620 + i, 128), oracle.normal(7630 + i, 128)
            q = oracle.normal(7640 + i, nh * hd)
            kn, vn = oracle.normal(7650 + i, nkv * hd), oracle.normal(7660 + i, nkv * hd)
            dq64, dkn64, dvn64 = ctx.upload(q64), ctx.upload(kn64), ctx.upload(vn64)
            dq, dkn, dvn = ctx.upload(q), ctx.upload(kn), ctx.upload(vn)
            ctx.layer_attention_devpos(dq64, dkn64, dvn64, dk64, dv64, dout64, 14, 2, 64, pos_dev, cap, 1e6,
                                       stream=s)
            ctx.layer_attention_devpos(dq, dkn, dvn, dkc, dvc, dout, nh, nkv, hd, pos_dev, cap, 1e6, stream=s)
            ctx.synchronize(s)
            assert int(pos_dev.numpy()[0]) == pos
            ref64, _, _ = oracle.layer_step(q64, kn64, vn64, k64, v64, 14, 2, 64, pos, 1e6)
            ref, _, _ = oracle.layer_step(q, kn, vn, kc, vc, nh, nkv, hd, pos, 1e6)
            assert_close(dout64.numpy(), ref64, f"head_dim 64 layer step at pos {pos}")
            assert_close(dout.numpy(), ref, f"layer {nh}/{nkv}/{hd} pos {pos} ({how})")
            assert ctx.check_device_error() == 0, f"device error at pos {pos}"
            for d in (dq64, dkn64, dvn64, dq, dkn, dvn):
                d.free()
        np.testing.assert_array_equal(dkc.numpy(), kc)
        np.testing.assert_array_equal(dvc.numpy(), vc)
        np.testing.assert_array_equal(dk64.numpy(), k64)
    finally:
        ctx.destroy_stream(s)
        for d in (dkc, dvc, dout, dk64, dv64, dout64, pos_dev):
            d.free()


def test_other_entry_points_refuse_other_shapes(ctx):
    U = tmac_attn.TMAC_ERR_UNSUPPORTED
    d = ctx.empty(1 << 16)
    p = d.ptr
    lib, h = ctx.lib, ctx.handle
    assert lib.tmac_attention_op(h, None, p, p, p, p, 14, 2, 63, 0) == U          # odd head_dim
    assert lib.tmac_attention_op(h, None, p, p, p, p, 2, 1, 258, 0) == U          # above 256
    assert lib.tmac_rope_op(h, None, p, 2, 63, 0, 1e6) == U
    assert lib.tmac_attention_decode_batched_kv(h, None, tmac_attn.TMAC_KV_BF16, p, p, p, p, 1, 14, 2, 128, 8,
                                                8) == U                            # narrow cache: head_dim 64 only
    assert lib.tmac_attention_decode_batched_kv(h, None, tmac_attn.TMAC_KV_Q8_0, p, p, p, p, 1, 3, 1, 64, 8,
                                                8) == U                            # narrow cache: compiled groups only
    assert lib.tmac_attention_prefill(h, None, p, p, p, p, 1, 4, 0, 4, 14, 2, 128) == U
    assert lib.tmac_attention_prefill(h, None, p, p, p, p, 1, 4, 0, 4, 3, 1, 64) == U
    assert lib.tmac_attention_decode_paged(h, None, tmac_attn.TMAC_KV_F32, p, p, p, 1, p, 1, p, p, 1, 3, 1, 64, 16,
                                           0) == U
    d.free()


@pytest.mark.parametrize("nh,nkv,hd", [(14, 2, 128), (12, 4, 96), (8, 8, 80), (5, 5, 256), (14, 2, 32), (20, 2, 64),
                                       (3, 1, 64), (2, 2, 4), (9, 3, 12), (9, 3, 66)])
@pytest.mark.parametrize("n_seq,max_len", [(1, 127), (1, 700), (3, 2050), (40, 300)])
def test_any_shape_splits(ctx, nh, nkv, hd, n_seq, max_len):
    """Batched, ragged and layer-step decode of shapes without compiled kernels, at lengths on and
    around the split, step and wave boundaries (splits are multiples of 32 rows from 128 rows on;
    heads 20 / 2 take two head tiles).  head_dim 66 keeps the unsplit row kernel."""
    k = oracle.normal(8000 + hd, (n_seq * max_len, nkv * hd))
    v = oracle.normal(8001 + hd, (n_seq * max_len, nkv * hd))
    q = oracle.normal(8002 + nh, (n_seq, nh * hd))
    offs = np.arange(n_seq, dtype=np.int64) * max_len
    lens = np.resize(np.array([max_len, 1, 0, 33, 128, 129, 255, 257, max_len - 1], np.int32), n_seq)
    lens = np.minimum(lens, max_len)
    dq, dk, dv, do, dl = (ctx.upload(x) for x in (q, k, v, offs, lens))
    dout = ctx.empty((n_seq, nh * hd))
    full = oracle.attention_ragged(q, k, v, offs, np.full(n_seq, max_len, np.int32), nh, nkv, hd, n_threads=8)
    dout.fill_bytes(0xFF)
    ctx.decode_batched(dq, dk, dv, dout, n_seq, nh, nkv, hd, max_len, max_len)
    assert_close(dout.numpy(), full, f"batched {nh}/{nkv}/{hd} {n_seq}x{max_len}")
    nz = lens > 0
    ref = np.zeros((n_seq, nh * hd), np.float32)
    ref[nz] = oracle.attention_ragged(q[nz], k, v, offs[nz], lens[nz], nh, nkv, hd, n_threads=8)
    for call in (ctx.decode_ragged, None):
        dout.fill_bytes(0xFF)
        if call:
            call(dq, dk, dv, do, dl, dout, n_seq, nh, nkv, hd, max_len)
        else:  # the partials in the fixed scratch array
            rc = ctx.lib.tmac_attention_decode_ragged_noalloc(ctx.handle, None, dq.ptr, dk.ptr, dv.ptr, do.ptr, dl.ptr,
                                                              dout.ptr, n_seq, nh, nkv, hd, max_len, 0)
            assert rc == tmac_attn.TMAC_OK
        assert_close(dout.numpy(), ref, f"ragged {nh}/{nkv}/{hd} {n_seq}x{max_len}")
    pos_dev = ctx.upload(np.zeros(1, np.int32))
    kn, vn = oracle.normal(8003, nkv * hd), oracle.normal(8004, nkv * hd)
    dkn, dvn = ctx.upload(kn), ctx.upload(vn)
    ctx.rope_prepare(hd, 1e6, max_len)
    kc, vc = k[:max_len].copy(), v[:max_len].copy()
    dkc, dvc = ctx.upload(kc), ctx.upload(vc)
    for pos in sorted({0, 31, 126, max_len // 2, max_len - 1}):
        ref1, _, _ = oracle.layer_step(q[0], kn, vn, kc, vc, nh, nkv, hd, pos, 1e6)
        if pos % 2:
            ctx.layer_attention(dq, dkn, dvn, dkc, dvc, dout, nh, nkv, hd, pos, max_len, 1e6)
        else:
            pos_dev.copy_from(np.array([pos], np.int32))
            ctx.layer_attention_devpos(dq, dkn, dvn, dkc, dvc, dout, nh, nkv, hd, pos_dev, max_len, 1e6)
        assert_close(dout.numpy()[0], ref1, f"layer {nh}/{nkv}/{hd} pos {pos} of {max_len}")
    np.testing.assert_array_equal(dkc.numpy(), kc)
    np.testing.assert_array_equal(dvc.numpy(), vc)
    for d in (dq, dk, dv, do, dl, dout, pos_dev, dkn, dvn, dkc, dvc):
        d.free()
    assert ctx.check_device_error() == 0


@pytest.mark.parametrize("nh,nkv,hd", [(14, 2, 128), (8, 8, 80), (9, 3, 66)])
@pytest.mark.parametrize("n_seq", [1, 6])
@pytest.mark.parametrize("noalloc", [False, True])
def test_any_shape_length_bound_is_exact(ctx, nh, nkv, hd, n_seq, noalloc):
    """A sequence one row longer than max_len gives NaN and error bit 1, whatever the number and
    length of the splits (1,000 rows: 7 splits of 160 at 14 / 2 heads), as does one of 2^31 - 1 rows.
    The rows behind the bound are allocated."""
    max_len, cap = 1000, 1152
    q = oracle.normal(8100, (n_seq, nh * hd))
    k, v = oracle.normal(8101, (n_seq * cap, nkv * hd)), oracle.normal(8102, (n_seq * cap, nkv * hd))
    lens = np.resize(np.array([max_len + 1, max_len, 3, 2**31 - 1, 0, max_len - 1], np.int32), n_seq)
    offs = np.arange(n_seq, dtype=np.int64) * cap
    dq, dk, dv, do, dl = (ctx.upload(x) for x in (q, k, v, offs, lens))
    dout = ctx.empty((n_seq, nh * hd))
    dout.fill_bytes(0x3F)
    if noalloc:
        rc = ctx.lib.tmac_attention_decode_ragged_noalloc(ctx.handle, None, dq.ptr, dk.ptr, dv.ptr, do.ptr, dl.ptr,
                                                          dout.ptr, n_seq, nh, nkv, hd, max_len, 0)
        assert rc == tmac_attn.TMAC_OK
    else:
        ctx.decode_ragged(dq, dk, dv, do, dl, dout, n_seq, nh, nkv, hd, max_len)
    got = dout.numpy()
    assert ctx.check_device_error() == tmac_attn.TMAC_ERR_DEVICE_FAULT
    for s in range(n_seq):
        if lens[s] > max_len:
            assert np.all(np.isnan(got[s])), f"sequence {s} of {lens[s]} rows"
        elif lens[s] == 0:
            assert np.all(got[s] == 0)
        else:
            ref = oracle.attention_ragged(q[s:s + 1], k, v, offs[s:s + 1], lens[s:s + 1], nh, nkv, hd, n_threads=8)
            assert_close(got[s:s + 1], ref, f"sequence {s} of {lens[s]} rows")
    for d in (dq, dk, dv, do, dl, dout):
        d.free()


@pytest.mark.parametrize("nh,nkv,hd", [(14, 2, 128), (5, 5, 256), (6, 3, 64), (9, 3, 66)])
def test_any_shape_infinite_rows(ctx, nh, nkv, hd):
    """An infinity in V reaches the output as an infinity, not as a NaN of a masked slot (0 * inf),
    also in the last row of a partial step and in the layer step's new row; a key that scores -inf
    weighs nothing, also where it is the only row of the last split (lengths 161, 321 and 801 of
    max_len 1,000, whose splits hold 160 rows at 14 / 2 heads)."""
    max_len, lens = 1000, np.array([161, 321, 801, 2, 999], np.int32)
    n_seq = lens.size
    offs = np.arange(n_seq, dtype=np.int64) * max_len
    q = np.abs(oracle.normal(8200, (n_seq, nh * hd))) + 0.1  # every head scores a key of -inf in dim 1 as -inf
    k, v = oracle.normal(8201, (n_seq * max_len, nkv * hd)), oracle.normal(8202, (n_seq * max_len, nkv * hd))
    last = offs + lens - 1
    ki, vi = k.copy(), v.copy()
    ki[last, 1::hd] = -np.inf
    vi[last, 0::hd] = np.inf
    dq, dk, dv, dki, dvi, do, dl = (ctx.upload(x) for x in (q, k, v, ki, vi, offs, lens))
    dout = ctx.empty((n_seq, nh * hd))
    ctx.decode_ragged(dq, dki, dv, do, dl, dout, n_seq, nh, nkv, hd, max_len)
    ref = oracle.attention_ragged(q, k, v, offs, lens - 1, nh, nkv, hd, n_threads=8)  # without the last row
    assert_close(dout.numpy(), ref, f"key of score -inf, {nh}/{nkv}/{hd}")
    ctx.decode_ragged(dq, dk, dvi, do, dl, dout, n_seq, nh, nkv, hd, max_len)
    got = dout.numpy()
    ref = oracle.attention_ragged(q, k, v, offs, lens, nh, nkv, hd, n_threads=8)
    first = np.arange(nh * hd) % hd == 0
    assert np.all(got[:, first] == np.inf)
    assert_close(got[:, ~first], ref[:, ~first], f"infinity in V, {nh}/{nkv}/{hd}")
    pos = 40
    kn, vn = oracle.normal(8203, nkv * hd), oracle.normal(8204, nkv * hd)
    vn[0::hd] = np.inf
    dkn, dvn = ctx.upload(kn), ctx.upload(vn)
    ctx.layer_attention(dq, dkn, dvn, dk, dv, dout, nh, nkv, hd, pos, max_len, 1e6)
    got = dout.numpy()[0]
    vn[0::hd] = 0
    ref, _, _ = oracle.layer_step(q[0], kn, vn, k[:max_len], v[:max_len], nh, nkv, hd, pos, 1e6)
    assert np.all(got[first] == np.inf)
    assert_close(got[~first], ref[~first], f"infinity in v_new, {nh}/{nkv}/{hd}")
    for d in (dq, dk, dv, dki, dvi, do, dl, dout, dkn, dvn):
        d.free()
    assert ctx.check_device_error() == 0


@pytest.mark.parametrize("nh,nkv,hd,cap", [(14, 2, 128, 1024), (14, 2, 128, 1025), (14, 2, 128, 4100), (12, 4, 96, 5000),
                                           (40, 8, 128, 2000), (9, 3, 12, 4096), (5, 5, 256, 513), (9, 3, 66, 2100)])
def test_layer_step_any_shape_large_capacity(ctx, nh, nkv, hd, cap):
    """The layer step under a device-side position at capacities on both sides of the one from which it is split
    (128 Ki floats of a kv head's rows), with 2 to 8 kv heads (the pairs of split and kv head are dealt to the
    XCDs) and several head tiles, at positions on the edges of runs and at the capacity's end."""
    kc, vc = oracle.normal(8300, (cap, nkv * hd)), oracle.normal(8301, (cap, nkv * hd))
    dkc, dvc, dout = ctx.upload(kc), ctx.upload(vc), ctx.empty(nh * hd)
    ctx.rope_prepare(hd, 1e6, cap)
    for i, pos in enumerate((0, 1, 255, 256, 511, cap // 2, cap - 1)):
        q, kn, vn = (oracle.normal(8310 + 3 * i + j, n * hd) for j, n in enumerate((nh, nkv, nkv)))
        dq, dkn, dvn, dpos = ctx.upload(q), ctx.upload(kn), ctx.upload(vn), ctx.upload(np.array([pos], np.int32))
        dout.fill_bytes(0xFF)
        ctx.layer_attention_devpos(dq, dkn, dvn, dkc, dvc, dout, nh, nkv, hd, dpos, cap, 1e6)
        ref, _, _ = oracle.layer_step(q, kn, vn, kc, vc, nh, nkv, hd, pos, 1e6)
        assert_close(dout.numpy(), ref, f"layer {nh}/{nkv}/{hd} pos {pos} of {cap}")
        for d in (dq, dkn, dvn, dpos):
            d.free()
    np.testing.assert_array_equal(dkc.numpy(), kc)
    np.testing.assert_array_equal(dvc.numpy(), vc)
    for d in (dkc, dvc, dout):
        d.free()
    assert ctx.check_device_error() == 0
