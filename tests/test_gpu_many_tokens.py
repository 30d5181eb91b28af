"""GPU: the many-token forms of the shared expert and the routers and the
grouped experts' work list, through the C ABI, at the sizes where a tile, a
grid, a piece or a dispatch rule ends."""
import ctypes

import numpy as np
import pytest

from oracle import binding as B

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nh():
    import nmoe_hip
    return nmoe_hip


@pytest.fixture(scope="module")
def ctx(nh):
    c = nh.Context(0, max_tokens=1100)
    yield c
    c.close()


def q4_tensor(rng, rows, cols, sigma, offset):
    """A q4 tensor whose biases are not -8 scale, and a device copy whose
    parts start `offset` elements into their buffers (w 4-byte, scales and
    biases 2-byte aligned)."""
    w = rng.integers(0, 2 ** 32, size=(rows, cols // 8), dtype=np.uint32)
    s = B.f32_to_bf16((rng.standard_normal((rows, cols // 64)) * sigma).astype(np.float32)).reshape(rows, -1)
    b = B.f32_to_bf16((rng.standard_normal((rows, cols // 64)) * 8 * sigma).astype(np.float32)).reshape(rows, -1)
    return w, s, b


def device_copy(ctx, t, offset):
    out = []
    for a in t:
        buf = ctx.alloc(a.nbytes + 16)
        buf.upload(a, offset * a.itemsize)
        out.append(buf.ptr + offset * a.itemsize)
    return tuple(out)


def dequant64(t):
    w, s, b = t
    q = ((w[..., None] >> (4 * np.arange(8, dtype=np.uint32))) & 15).reshape(s.shape[0], s.shape[1], 64)
    f = lambda v: B.bf16_to_f32(v).reshape(v.shape).astype(np.float64)
    return (q * f(s)[..., None] + f(b)[..., None]).reshape(s.shape[0], -1)


def tokens(rng, ctx, nh, xdt, ntok):
    x = rng.standard_normal((ntok, 2048)).astype(np.float32)
    if xdt == "f32":
        return x, ctx.to_device(x), nh.F32
    xb = B.f32_to_bf16(x)
    return B.bf16_to_f32(xb).reshape(ntok, 2048), ctx.to_device(xb), nh.BF16


# per-token kernels up to 35 tokens (1, 2 or 4 tokens a block); then 16-, 32-
# and 64-token tiles, each with a ragged last tile and, for the largest, the
# die-wise tile order (16 tiles and more)
@pytest.mark.parametrize("xdt,ntok", [("f32", 4), ("bf16", 5), ("f32", 13), ("bf16", 35), ("f32", 36), ("bf16", 241),
                                      ("f32", 257), ("bf16", 512), ("f32", 513), ("bf16", 1025)])
def test_shared_expert_many_tokens(ctx, nh, xdt, ntok):
    """shared_out and the score against the products in 64 bits (relative L2
    within 1e-6: fp32 sums of 2,048 and 512 terms, each rounding 2^-24, stay
    below 5e-7), a few tokens against the oracle, every token's score bit for
    bit the per-token kernels', and nothing written past the last token."""
    rng = np.random.default_rng(1000 + ntok)
    t = {n: q4_tensor(rng, r, c, s, 1) for n, (r, c, s) in
         {"gate": (512, 2048, 0.004), "up": (512, 2048, 0.004), "down": (2048, 512, 0.008),
          "score": (1, 2048, 0.004)}.items()}
    desc = nh.Context.shared_expert_desc(*(device_copy(ctx, t[n], 1) for n in ("gate", "up", "down", "score")))
    x, dx, dt = tokens(rng, ctx, nh, xdt, ntok)
    guard = np.full(2048, 7.5, np.float32)
    so, gr = ctx.alloc((ntok + 1) * 8192), ctx.alloc((ntok + 1) * 4)
    so.upload(guard, ntok * 8192)
    gr.upload(guard[:1], ntok * 4)
    ctx._check(ctx.shared_expert(desc, dx, dt, ntok, so, gr))
    got, got_g = so.download(np.float32, (ntok + 1, 2048)), gr.download(np.float32, ntok + 1)
    assert np.array_equal(got[ntok], guard) and got_g[ntok] == 7.5
    x64 = x.astype(np.float64)
    g, u = x64 @ dequant64(t["gate"]).T, x64 @ dequant64(t["up"]).T
    want = (g / (1 + np.exp(-g)) * u) @ dequant64(t["down"]).T
    want_g = (x64 @ dequant64(t["score"]).T)[:, 0]
    rel = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)
    print(f"[shared] {xdt} {ntok} tokens: rel {rel(got[:ntok], want):.2e}, score {rel(got_g[:ntok], want_g):.2e}")
    assert rel(got[:ntok], want) < 1e-6 and rel(got_g[:ntok], want_g) < 1e-6
    pick = np.unique([0, ntok // 2, ntok - 1])
    want_so, want_gr = B.shared_expert({n: t[n] for n in t}, x[pick])
    assert rel(got[pick], want_so) < 2e-6 and rel(got_g[pick], want_gr) < 2e-6
    few = ctx.alloc(ntok * 4)
    for t0 in range(0, ntok, 32):
        ctx._check(ctx.shared_expert(desc, dx.ptr + t0 * 2048 * (4 if dt == nh.F32 else 2), dt, min(32, ntok - t0), so,
                                     few.ptr + 4 * t0))
    np.testing.assert_array_equal(got_g[:ntok].view(np.uint32), few.download(np.uint32, ntok))


@pytest.mark.parametrize("xdt,ntok", [("f32", 67), ("bf16", 300)])
def test_shared_expert_place_in_the_call(ctx, nh, xdt, ntok):
    """A token's matrix-form output does not depend on its place in the call:
    the tokens from the first, second, fourth and eighteenth on, bit for bit."""
    rng = np.random.default_rng(ntok)
    t = [q4_tensor(rng, r, k, s, 1) for r, k, s in
         ((512, 2048, 0.004), (512, 2048, 0.004), (2048, 512, 0.008), (1, 2048, 0.004))]
    desc = nh.Context.shared_expert_desc(*(device_copy(ctx, q, 1) for q in t))
    _, dx, dt = tokens(rng, ctx, nh, xdt, ntok)
    got = []
    for first in (0, 1, 3, 17):
        n = ntok - first
        so, gr = ctx.alloc(n * 8192), ctx.alloc(n * 4)
        ctx._check(ctx.shared_expert(desc, dx.ptr + first * 2048 * (4 if dt == nh.F32 else 2), dt, n, so, gr))
        got.append((so.download(np.uint32, (n, 2048))[17 - first:], gr.download(np.uint32, n)[17 - first:]))
    for so, gr in got[1:]:
        np.testing.assert_array_equal(so, got[0][0])
        np.testing.assert_array_equal(gr, got[0][1])


@pytest.mark.parametrize("xdt,ntok", [("f32", 16389), ("bf16", 16428)])
def test_shared_expert_chunks(nh, xdt, ntok):
    """A call of more tokens than the matrix-core launches take at a time: the
    tokens around the seam, and the last ones, bit for bit those of a short
    call's matrix form; the score of the first tokens bit for bit the
    per-token kernels'; nothing written past the last token."""
    rng = np.random.default_rng(ntok)
    with nh.Context(0, max_tokens=ntok) as c:
        t = [q4_tensor(rng, r, k, s, 1) for r, k, s in
             ((512, 2048, 0.004), (512, 2048, 0.004), (2048, 512, 0.008), (1, 2048, 0.004))]
        desc = nh.Context.shared_expert_desc(*(device_copy(c, q, 1) for q in t))
        _, dx, dt = tokens(rng, c, nh, xdt, ntok)
        row = 8192 if dt == nh.F32 else 4096

        def run(first, n):
            so, gr = c.to_device(np.full((n + 1, 2048), 7.5, np.float32)), c.to_device(np.full(n + 1, 7.5, np.float32))
            c._check(c.shared_expert(desc, dx.ptr + first * row, dt, n, so, gr))
            so, gr = so.download(np.uint32, (n + 1, 2048)), gr.download(np.uint32, n + 1)
            assert (so[n].view(np.float32) == 7.5).all() and gr[n:].view(np.float32)[0] == 7.5
            return so[:n], gr[:n]

        so, gr = run(0, ntok)
        for first, n in ((0, 36), (ntok - 97, 97), (ntok - 44, 44)):
            part, pg = run(first, n)
            np.testing.assert_array_equal(so[first:first + n], part)
            np.testing.assert_array_equal(gr[first:first + n], pg)
        np.testing.assert_array_equal(gr[:35], run(0, 35)[1])


def test_context_scratch_of_many_tokens(nh):
    """What a context takes a token beyond 16,384: the routed experts' scratch
    (108,132 bytes), none for the shared expert, whose own is bounded."""
    path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l) if nh.lib() else None
    hip = ctypes.CDLL(path)

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    used = []
    for n in (16384, 65536):
        c = nh.Context(0, max_tokens=n)
        after = free()
        c.close()
        used.append(free() - after)
    per = (used[1] - used[0]) / (65536 - 16384)
    print(f"[scratch] {used} bytes, {per:.0f} a token")
    assert per < 108132 + 1000  # the allocations' granules


# one row a wavefront for few terms, then tiles of 16 x 16, 32 x 32 (from 513
# tokens) and 32 x 64 (from 1,025), with ragged last tiles of tokens and experts:
# either side of each line of the rule, for few experts too
@pytest.mark.parametrize("kind,xdt,ntok,ne", [
    ("bf16", "f32", 96, 256), ("bf16", "bf16", 241, 250), ("bf16", "f32", 257, 256), ("bf16", "bf16", 290, 33),
    ("bf16", "bf16", 1025, 256), ("bf16", "f32", 1041, 241), ("q4", "f32", 192, 256), ("q4", "bf16", 193, 256),
    ("q4", "f32", 300, 17), ("q4", "bf16", 1025, 250), ("bf16", "bf16", 104, 256), ("bf16", "bf16", 512, 256),
    ("bf16", "f32", 513, 256), ("bf16", "bf16", 1100, 33), ("bf16", "f32", 1100, 120), ("q4", "f32", 208, 256),
    ("q4", "f32", 257, 256), ("q4", "f32", 384, 256), ("q4", "bf16", 200, 256), ("q4", "bf16", 384, 250),
    ("q4", "f32", 1000, 40), ("q4", "bf16", 1100, 40)])
def test_router_many_tokens_bit_exact(ctx, nh, kind, xdt, ntok, ne):
    """The matrix form's logits bit for bit the few-token kernel's (the same
    tokens 64 at a time) and, for a few tokens, the oracle's; subnormal, huge,
    infinite and NaN tokens among them; nothing written past the last logit."""
    rng = np.random.default_rng(ntok * 7 + ne)
    if kind == "bf16":
        w = B.f32_to_bf16((rng.standard_normal((ne, 2048)) * 0.02).astype(np.float32)).reshape(ne, 2048)
        r = nh.Context.router_bf16(ctx.to_device(w), ne)
    else:
        t = q4_tensor(rng, ne, 2048, 0.004, 1)
        r = nh.Context.router_q4(*device_copy(ctx, t, 1), ne)
    x = rng.standard_normal((ntok, 2048)).astype(np.float32)
    x[1] *= np.float32(1e-38)
    x[2] *= np.float32(3e36)
    x[3, 17], x[4, 900], x[5] = np.inf, np.nan, 0.0
    if xdt == "bf16":
        xb = B.f32_to_bf16(x)
        x, dx, dt, size = B.bf16_to_f32(xb).reshape(ntok, 2048), ctx.to_device(xb), nh.BF16, 2
    else:
        dx, dt, size = ctx.to_device(x), nh.F32, 4
    lg, ref = ctx.alloc(ntok * ne * 4 + 64), ctx.alloc(ntok * ne * 4)
    lg.upload(np.full(16, 7.5, np.float32), ntok * ne * 4)
    ctx._check(ctx.router_logits(r, dx, dt, ntok, lg))
    for t0 in range(0, ntok, 64):
        ctx._check(ctx.router_logits(r, dx.ptr + t0 * 2048 * size, dt, min(64, ntok - t0), ref.ptr + t0 * ne * 4))
    got, want = lg.download(np.float32, (ntok, ne)), ref.download(np.float32, (ntok, ne))
    assert np.array_equal(lg.download(np.float32, 16, ntok * ne * 4), np.full(16, 7.5, np.float32))
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fine = ~np.isnan(want)
    np.testing.assert_array_equal(got.view(np.uint32)[fine], want.view(np.uint32)[fine])
    for tok in (0, 16, ntok - 1):
        if kind == "bf16":
            o = B.router_logits_bf16(w, x[tok])
        else:
            o, xt = np.zeros(ne, np.float32), np.ascontiguousarray(x[tok], np.float32)
            B.oracle().orc_router_logits_q4(t[0].ctypes.data, t[1].ctypes.data, t[2].ctypes.data, xt.ctypes.data, ne,
                                            2048, o.ctypes.data)
        np.testing.assert_array_equal(got[tok].view(np.uint32), o.view(np.uint32))


# the q4 terms' products at the ends of the exponent range, a 16 x 16 tile for
# each: scales around 2 (s x overflows for the largest x), around 1e37 (q s
# overflows) and below 2^-63 down to subnormals, with zero codes and scales and
# biases of either sign; scales below 1 with the same x
@pytest.mark.parametrize("xdt,ntok", [("bf16", 208), ("f32", 224)])
def test_router_q4_extreme_products(ctx, nh, xdt, ntok):
    """Bit for bit the few-token kernel's logits (NaN for NaN) and the oracle's."""
    rng = np.random.default_rng(ntok)
    w, s, b = q4_tensor(rng, 256, 2048, 2.0, 1)
    w[::7] &= np.uint32(0x0F0F0F0F)  # half of the row's codes 0
    f = B.bf16_to_f32(s).reshape(s.shape).copy()
    for e, m in enumerate((1.0, 1e37, 1e-20, 1e-30, 1e-38)):
        f[16 * e:16 * e + 16] = np.clip(f[16 * e:16 * e + 16], -8, 8) * np.float32(m)
    f[80:96, ::5] = 0.0
    f[96:128] = np.clip(f[96:128] * np.float32(0.2), -1, 1)
    b = np.where(rng.random(s.shape) < 0.5, -8 * f.astype(np.float64), np.where(rng.random(s.shape) < 0.5, 0.0, f))
    s, b = (B.f32_to_bf16(np.clip(v, -3e38, 3e38).astype(np.float32)).reshape(s.shape) for v in (f, b))
    r = nh.Context.router_q4(*device_copy(ctx, (w, s, b), 1), 256)
    x = rng.standard_normal((ntok, 2048)).astype(np.float32)
    for t, m in enumerate((1e37, 8e37, 3e36, 1e20, 1.0, 1e-5, 1e-20, 1e-25, 1e-37, 1e-38)):
        x[16 * t:16 * t + 16] = np.clip(x[16 * t:16 * t + 16], -4, 4) * np.float32(m)
    x[0], x[1], x[2], x[16, ::3] = 3.3e38, 0.0, 0.0, 0.0
    x[1, 77], x[2, 900] = 3e38, -1e38  # one term only: no other sign makes a NaN of an infinity
    if xdt == "bf16":
        xb = B.f32_to_bf16(x)
        x, dx, dt, size = B.bf16_to_f32(xb).reshape(ntok, 2048), ctx.to_device(xb), nh.BF16, 2
    else:
        dx, dt, size = ctx.to_device(x), nh.F32, 4
    assert np.isfinite(x).all() and np.isfinite(B.bf16_to_f32(s)).all() and np.isfinite(B.bf16_to_f32(b)).all()
    lg, ref = ctx.alloc(ntok * 1024), ctx.alloc(ntok * 1024)
    ctx._check(ctx.router_logits(r, dx, dt, ntok, lg))
    for t0 in range(0, ntok, 64):
        ctx._check(ctx.router_logits(r, dx.ptr + t0 * 2048 * size, dt, min(64, ntok - t0), ref.ptr + t0 * 1024))
    got, want = lg.download(np.float32, (ntok, 256)), ref.download(np.float32, (ntok, 256))
    assert np.isnan(want).any() and np.isinf(want).any() and np.isfinite(want).any()
    for t in list(range(0, ntok, 16)) + [1, 2, ntok - 1]:
        o, xt = np.zeros(256, np.float32), np.ascontiguousarray(x[t], np.float32)
        B.oracle().orc_router_logits_q4(w.ctypes.data, s.ctypes.data, b.ctypes.data, xt.ctypes.data, 256, 2048,
                                        o.ctypes.data)
        np.testing.assert_array_equal(want[t], o)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    fine = ~np.isnan(want)
    np.testing.assert_array_equal(got.view(np.uint32)[fine], want.view(np.uint32)[fine])


# entries an expert gets: either side of a 16-entry row block and of one, two
# and three 64-entry pieces; one expert only; few experts of many pieces, on
# either side of the most entries one launch takes (8,192); every expert with
# a piece of 32, the most pieces of more than 16 entries.  A third of the
# tokens also have an entry on an expert of few entries; slots left over hold
# indexes outside the layer
@pytest.mark.parametrize("bits,xdt,counts,ntok", [
    (4, "f32", [63, 64, 65, 127, 128, 129, 16, 17, 1, 2], 129), (2, "bf16", [64, 128, 192, 193, 15, 48, 49], 193),
    (4, "bf16", [200], 200), (2, "f32", [1025, 1024, 961, 960, 449], 1025), (4, "bf16", [1024, 1000, 961, 449], 1024),
    (4, "f32", [32] * 256, 1024), (2, "bf16", [32] * 256, 1024)])
def test_grouped_pieces(nh, bits, xdt, counts, ntok):
    """The grouped path (in one launch, up to 8,192 entries, and in two: the
    same bits) against the per-token kernels of the same call, relative L2
    within 1e-4 as the path's act planes (2^-17 a term) and fp32 sums allow,
    every token held to 1e-3, and nothing written past the last token."""
    rng = np.random.default_rng(len(counts) + ntok)
    slots = np.full((ntok, 8), 0xFFFFFFFF, np.uint32)
    fill = np.zeros(ntok, int)
    for e, n in enumerate(counts):  # expert 11 e mod 256: n different tokens, the emptiest first
        for t in np.argsort(fill + rng.random(ntok) * 0.5)[:n]:
            slots[t, fill[t]] = 11 * e % 256
            fill[t] += 1
    if len(counts) > 1:
        for t in range(0, ntok, 3):
            if fill[t] < 8:
                slots[t, fill[t]] = 100 + t % 150
    w = rng.dirichlet(np.ones(8), size=ntok).astype(np.float32)
    c = nh.Context(0, max_tokens=ntok)
    try:
        c.synth_layer(1, bits, 5, 0.02 if bits == 4 else 0.05)
        x, dx, dt = tokens(rng, c, nh, xdt, ntok)
        h = rng.standard_normal((ntok, 2048)).astype(np.float32)
        di, dw, dh = c.to_device(slots), c.to_device(w), c.to_device(h)
        got = []
        for gmin, one in ((8, True), (8, False), (1 << 20, True)):
            c.set_grouped_min_tokens(gmin)
            if not c.set_grouped_one_launch(one) and one and gmin == 8:
                continue
            out = c.to_device(np.full((ntok + 1, 2048), 7.5, np.float32))
            c._check(c.experts(bits, 1, dx, dt, ntok, 8, di, dw, dh, out))
            o = out.download(np.float32, (ntok + 1, 2048))
            assert (o[ntok] == 7.5).all()
            got.append(o[:ntok].astype(np.float64) - h)
        assert c.device_status() == nh.OK
        # a wrong tile count fails a call in one launch alone: which of the forms ran above
        c.set_grouped_min_tokens(8)
        if c.set_grouped_one_launch(True):
            assert len(got) == 3
            c._check(c.set_option(nh.OPT_SKEW_TILES, 0))
            c._check(c.experts(bits, 1, dx, dt, ntok, 8, di, dw, dh, out))
            assert c.device_status() == (nh.ETIMEDOUT if ntok * 8 <= 8192 else nh.OK)
    finally:
        c.close()
    want = got.pop()
    for o in got:
        np.testing.assert_array_equal(o, got[0])
    rel = np.linalg.norm(got[0] - want, axis=1) / np.maximum(np.linalg.norm(want, axis=1), 1e-6)
    print(f"[pieces] q{bits} {xdt} {ntok} tokens: worst token {rel.max():.2e}")
    assert np.linalg.norm(got[0] - want) / np.linalg.norm(want) < 1e-4 and rel.max() < 1e-3
