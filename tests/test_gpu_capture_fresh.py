"""Calls captured on a context that has run nothing before: the schedules that keep partials between
two launches (any-shape splits, prefill key runs) depend on the shape alone, so the captured calls
give the bits of eager ones, on every replay, also after the context's workspace has grown.

Shapes whose partials are the largest: 64 heads over 8 kv heads of 256 dims (64 splits), 100 queries
after 4,000 rows (17 stages, all runs of one).  Oracle: tmac_gguf.cpp:1093-1128."""
import numpy as np
import pytest

import oracle
import tmac_attn
from conftest import assert_close

pytestmark = pytest.mark.gpu
HD, QD, KVD = 64, 14 * 64, 2 * 64


def bf16_round(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32)


@pytest.mark.parametrize("kind", ["any", "any_layer", "prefill", "prefill_tiles"])
def test_capture_on_a_fresh_context(kind):
    with tmac_attn.Context(0) as ctx:
        s = ctx.stream()
        if kind in ("any", "any_layer"):
            nh, nkv, hd, rows = 64, 8, 256, 8192
            q = oracle.normal(9500, (1, nh * hd))
            k, v = oracle.normal(9501, (rows, nkv * hd)), oracle.normal(9502, (rows, nkv * hd))
            dk, dv = ctx.upload(k), ctx.upload(v)
            dq, dout = ctx.upload(q), ctx.empty((1, nh * hd))
            if kind == "any":
                def call():
                    ctx.decode_batched(dq, dk, dv, dout, 1, nh, nkv, hd, rows, rows, stream=s)
                ref = oracle.attention_ragged(q, k, v, np.zeros(1, np.int64), np.array([rows], np.int32), nh, nkv, hd,
                                              n_threads=8)
            else:
                kn, vn = oracle.normal(9503, nkv * hd), oracle.normal(9504, nkv * hd)
                dkn, dvn, dpos = ctx.upload(kn), ctx.upload(vn), ctx.upload(np.array([5000], np.int32))
                ctx.rope_prepare(hd, 1e6, rows)

                def call():
                    ctx.layer_attention_devpos(dq, dkn, dvn, dk, dv, dout, nh, nkv, hd, dpos, rows, 1e6, stream=s)
                ref = oracle.layer_step(q[0], kn, vn, k, v, nh, nkv, hd, 5000, 1e6)[0][None]
        else:
            n_q, prefix = 100, 4000
            rows = n_q + prefix
            q = bf16_round(oracle.normal(9510, (1, n_q, QD)))
            k, v = (bf16_round(oracle.normal(9511 + i, (1, rows, KVD))) for i in range(2))
            dq, dk, dv, dout = ctx.upload(q), ctx.upload(k), ctx.upload(v), ctx.empty(q.shape)
            if kind == "prefill":
                def call():
                    ctx.prefill(dq, dk, dv, dout, 1, n_q, prefix, rows, 14, 2, HD, stream=s)
            else:
                tiles = ctx.empty(ctx.prefill_tiles_bytes(1, 2, rows) // 4)

                def call():
                    ctx.prefill_pack_rows(dk, dv, rows, tiles, rows, 1, 2, HD, 0, rows, stream=s)
                    ctx.prefill_tiles(dq, tiles, rows, dout, 1, n_q, prefix, 14, 2, HD, stream=s)
            ref = oracle.prefill(q, k, v, 1, n_q, prefix, rows, 14, 2, HD, n_threads=8).reshape(q.shape)
        ctx.synchronize(None)
        ctx.step_begin(s)
        call()
        g = ctx.step_end(s)
        got = []
        for replay in range(4):
            dout.fill_bytes(0xFF, stream=s)
            if replay == 2:
                call()  # eagerly
            else:
                ctx.graph_launch(g, s)
            ctx.synchronize(s)
            got.append(dout.numpy())
            if replay == 0:  # a call that needs a larger workspace (2 x 4,000 rows of prefill tiles, all key runs)
                x = ctx.empty((2, 4000, KVD))
                x.fill_bytes(0, stream=s)
                y = ctx.empty((2, 2000, QD))
                y.fill_bytes(0, stream=s)
                ctx.prefill(y, x, x, y, 2, 2000, 2000, 4000, 14, 2, HD, stream=s)
                ctx.synchronize(s)
        assert_close(got[0], ref, kind)
        for i, r in enumerate(got[1:]):
            np.testing.assert_array_equal(r.view(np.uint32), got[0].view(np.uint32), err_msg=f"{kind}, pass {i + 1}")
        assert ctx.check_device_error() == 0
        ctx.graph_destroy(g)
        ctx.destroy_stream(s)
