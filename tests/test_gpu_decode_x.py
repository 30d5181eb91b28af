"""GPU: one token through the fused launch with x given (each type of x and
code width, routed inside the launch and with the routing given), and the
per-token kernels of a few tokens."""
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


@pytest.mark.parametrize("bits,k,ntok", [(4, 1, 2), (4, 6, 7), (4, 7, 3), (2, 1, 7), (2, 6, 3), (2, 8, 7),
                                         (4, 2, 7), (4, 3, 5), (2, 2, 5), (2, 3, 2)])
def test_few_tokens_unused_slots(bits, k, ntok):
    """The per-token kernels: slots past k hold indexes outside the layer and
    NaN weights, one used slot an index outside the layer (weight 0); x, idx
    and w lie between values that would show in the output."""
    import nmoe_hip as nh
    rng = np.random.default_rng(70 + bits + k + ntok)
    seed, layer = 9, 2
    esz = B.EXPERT_SIZE[bits]
    idx = np.full((ntok, 8), 0xFFFFFFFF, np.uint32)
    for t in range(ntok):
        idx[t, :k] = rng.choice(256, k, replace=False)
    w = np.full((ntok, 8), np.nan, np.float32)
    w[:, :k] = rng.dirichlet(np.ones(k), size=ntok).astype(np.float32)
    pack = np.zeros(B.EXPERTS * esz, np.uint8)
    for e in set(idx[:, :k].ravel().tolist()):
        pack[e * esz:(e + 1) * esz] = B.syn_expert(bits, seed, layer, e, SIGMA[bits])
    xb = B.f32_to_bf16(rng.standard_normal((ntok, 2048)).astype(np.float32)).reshape(ntok, 2048)
    x = B.bf16_to_f32(xb).reshape(ntok, 2048)
    h = rng.standard_normal((ntok, 2048)).astype(np.float32)
    ow, oi = w.copy(), idx.copy()
    ow[:, k:], oi[:, k:] = 0.0, 0
    if k > 1:
        idx[ntok - 1, k - 1] = 256
        ow[ntok - 1, k - 1] = 0.0
    want = B.moe_experts(pack, bits, x, k, oi, ow, h)
    c = nh.Context(0, max_tokens=8)
    try:
        c.synth_layer(layer, bits, seed, SIGMA[bits])
        di, dw, dh = c.to_device(idx), c.to_device(w), c.to_device(h)
        for arr, dt in ((x, nh.F32), (xb, nh.BF16)):
            pad = np.full(8, np.nan, np.float32) if dt == nh.F32 else np.full(8, 0x7FC0, np.uint16)
            dx = c.to_device(np.concatenate([pad, arr.ravel(), pad]))
            out = c.to_device(np.full((ntok + 1, 2048), 7.5, np.float32))
            c._check(c.experts(bits, layer, dx.ptr + pad.nbytes, dt, ntok, k, di, dw, dh, out))
            got = out.download(np.float32, (ntok + 1, 2048))
            assert_close(got[:ntok], want, what=f"q{bits} k={k} ntok={ntok} dt={dt}")
            assert (got[ntok] == 7.5).all()
    finally:
        c.close()
