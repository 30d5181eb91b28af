"""GPU: one token through the fused launch with x given, each type of x and
code width, routed inside the launch and with the routing given."""
import numpy as np
import pytest

from conftest import assert_close
from oracle import binding as B

pytestmark = pytest.mark.gpu
SIGMA = {4: 0.004, 2: 0.016}


@pytest.mark.parametrize("bits,k", [(4, 8), (4, 1), (2, 8), (2, 6)])
def test_given_x_types_agree(bits, k):
    """x between NaN neighbours, as fp32 and as the same values in bf16: the
    same bits out of either (both run on the fp32 values), the oracle's
    routing bit for bit and its output within the path's tolerance."""
    import nmoe_hip as nh
    rng = np.random.default_rng(60 + bits + k)
    seed, layer = 7, 3
    W = B.syn_bf16(256 * 2048, seed, layer, 16, 0.02).reshape(256, 2048)
    xb = B.f32_to_bf16(rng.standard_normal(2048).astype(np.float32))
    x = B.bf16_to_f32(xb).reshape(1, 2048)
    h = rng.standard_normal((1, 2048)).astype(np.float32)
    oi, ow, _ = B.route(B.router_logits_bf16(W, x[0]), k)
    esz = B.EXPERT_SIZE[bits]
    pack = np.zeros(B.EXPERTS * esz, np.uint8)
    for e in set(oi[:k].tolist()):
        pack[e * esz:(e + 1) * esz] = B.syn_expert(bits, seed, layer, e, SIGMA[bits])
    want = B.moe_experts(pack, bits, x, k, oi[None], ow[None], h)
    c = nh.Context(0, max_tokens=4)
    try:
        c.synth_layer(layer, bits, seed, SIGMA[bits])
        router, dh, outs = c.router_bf16(c.to_device(W)), c.to_device(h), []
        out, idx, w, lg = c.alloc(8192), c.alloc(32), c.alloc(32), c.alloc(1024)
        for arr, dt in ((x.astype(np.float32).ravel(), nh.F32), (xb.ravel(), nh.BF16)):
            pad = np.full(8, np.nan, np.float32) if dt == nh.F32 else np.full(8, 0x7FC0, np.uint16)
            dx = c.to_device(np.concatenate([pad, arr, pad]))
            c._check(c.moe_layer(layer, router, dx.ptr + pad.nbytes, dt, 1, k, dh, out, idx, w, lg))
            np.testing.assert_array_equal(idx.download(np.uint32, 8)[:k], oi[:k])
            np.testing.assert_array_equal(w.download(np.float32, 8)[:k].view(np.uint32), ow[:k].view(np.uint32))
            outs.append(out.download(np.float32, (1, 2048)))
            c._check(c.experts(bits, layer, dx.ptr + pad.nbytes, dt, 1, k, idx, w, dh, out))
            outs.append(out.download(np.float32, (1, 2048)))
        assert c.device_status() == nh.OK
    finally:
        c.close()
    assert_close(outs[0], want, what=f"q{bits} k={k}")
    for o in outs[1:]:
        np.testing.assert_array_equal(o.view(np.uint32), outs[0].view(np.uint32))
