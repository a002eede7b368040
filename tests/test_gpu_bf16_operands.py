"""Products whose operands are read as bf16 from memory (nchip_gemm_bf16_operands, the grouped
launch with precision 2, nchip_cast_bf16) and the shadow copies that feed them at the tensor
level.  The yardstick is numpy: both operands rounded to bf16 (nearest even, the rounding
tests/test_oracle_ops.py pins against torch), products and sums in float64 - the kernels
accumulate the same rounded values in fp32, so they must agree to fp32 summation error (1e-5
of the largest magnitude); bf16 copies of results must be the nearest-even rounding of the
fp32 results, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from conftest import hip_lib_path

pytestmark = pytest.mark.gpu


def bf16_round(x):
    """float32 -> the float32 value of its nearest-even bf16 rounding, and the 16 bits"""
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32).astype(np.uint64)
    r = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint32)
    return (r << 16).view(np.float32).reshape(np.shape(x)), r.astype(np.uint16).reshape(np.shape(x))


def relerr(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.abs(a - b).max() / (np.abs(b).max() + 1e-30))


class Args(C.Structure):
    _fields_ = [("ta", C.c_int), ("tb", C.c_int), ("m", C.c_int), ("n", C.c_int), ("k", C.c_int),
                ("alpha", C.c_float), ("A16", C.c_void_p), ("B16", C.c_void_p), ("lda", C.c_int64),
                ("ldb", C.c_int64), ("C", C.c_void_p), ("ldc", C.c_int64), ("C16", C.c_void_p),
                ("bias", C.c_void_p), ("act", C.c_int), ("pre", C.c_void_p), ("addend", C.c_void_p),
                ("dpre", C.c_void_p), ("dact", C.c_int), ("rowsum", C.c_void_p), ("rows_written", C.POINTER(C.c_int))]


class Problem(C.Structure):
    _fields_ = [("A", C.c_void_p), ("B", C.c_void_p), ("C", C.c_void_p), ("A2", C.c_void_p), ("B2", C.c_void_p),
                ("m", C.c_int), ("n", C.c_int), ("k", C.c_int), ("k2", C.c_int),
                ("lda", C.c_int), ("ldb", C.c_int), ("ldc", C.c_int), ("tile_start", C.c_int), ("alpha", C.c_float)]


@pytest.fixture()
def raw(hip, pkg):
    lib = C.CDLL(hip_lib_path(pkg))
    lib.nchip_cast_bf16.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int64]
    lib.nchip_gemm_bf16_operands.argtypes = [C.c_void_p, C.POINTER(Args)]
    lib.nchip_gemm_grouped.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_double]
    st = C.c_void_p(hip.nc_context_stream(hip.ctx))
    ptr = lambda t: C.c_void_p(hip.lib.nc_tensor_get_ptr(t, None))
    return lib, st, ptr


def gelu(x):
    return 0.5 * x * (1.0 + np.tanh(0.7978845608 * (x + 0.044715 * x ** 3)))


def gelu_grad(x):
    c0, c1 = 0.7978845608, 0.044715
    t = np.tanh(c0 * (x + c1 * x ** 3))
    return 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * c0 * (1 + 3 * c1 * x * x)


@pytest.mark.parametrize("n", [8, 4096, 1000003, 13])
def test_cast_is_round_to_nearest_even(hip, raw, rng, n):
    lib, st, ptr = raw
    x = (rng.standard_normal(n) * np.exp(rng.uniform(-30, 30, n))).astype(np.float32)
    x[: min(n, 6)] = np.array([0.0, -0.0, 1.00390625, 1.01171875, np.float32(2.0 ** -130), 3.0e38], np.float32)[: min(n, 6)]
    src, dst = hip.tensor(x), hip.tensor(np.zeros(n, np.uint16))
    assert lib.nchip_cast_bf16(st, ptr(src), ptr(dst), n) == 0
    got = hip.numpy(dst)
    hip.free(src, dst)
    assert np.array_equal(got, bf16_round(x)[1])


# (m, n, k): every tile class (forced below) must divide what it needs whole
SHAPES = [(128, 128, 64), (256, 192, 128), (512, 2048, 512), (384, 100, 192), (128, 77, 64), (1024, 256, 320)]


@pytest.mark.parametrize("cls", [0, 1, 2, 3])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_product_from_bf16_operands(hip, raw, rng, m, n, k, ta, tb, cls):
    lib, st, ptr = raw
    a = rng.standard_normal((m, k) if ta else (k, m)).astype(np.float32)      # numpy order: (columns, rows)
    b = rng.standard_normal((k, n) if tb else (n, k)).astype(np.float32)
    bias = rng.standard_normal(m).astype(np.float32)
    add = rng.standard_normal((n, m)).astype(np.float32)
    A = bf16_round(a)[0].astype(np.float64)
    B = bf16_round(b)[0].astype(np.float64)
    Am = A if not ta else A.T                  # (k, m) numpy = column-major (m, k)
    Bm = B if not tb else B.T                  # (n, k)
    pre = 0.75 * (Bm @ Am) + bias              # (n, m): column-major (m, n)
    want = gelu(pre) + add
    t = {k_: hip.tensor(v) for k_, v in dict(a=a, b=b, bias=bias, add=add).items()}
    t.update(a16=hip.tensor(np.zeros(a.shape, np.uint16)), b16=hip.tensor(np.zeros(b.shape, np.uint16)),
             c=hip.tensor(np.full((n, m), 7.0, np.float32)), pre=hip.tensor(np.full((n, m), 7.0, np.float32)),
             c16=hip.tensor(np.full((n, m), 7, np.uint16)))
    assert lib.nchip_cast_bf16(st, ptr(t["a"]), ptr(t["a16"]), a.size) == 0
    assert lib.nchip_cast_bf16(st, ptr(t["b"]), ptr(t["b16"]), b.size) == 0
    lib.nchip_gemm_bf16_operands_class(cls)
    g = Args(ta=ta, tb=tb, m=m, n=n, k=k, alpha=0.75, A16=ptr(t["a16"]), B16=ptr(t["b16"]),
             lda=k if ta else m, ldb=n if tb else k, C=ptr(t["c"]), ldc=m, C16=ptr(t["c16"]),
             bias=ptr(t["bias"]), act=1, pre=ptr(t["pre"]), addend=ptr(t["add"]))
    rc = lib.nchip_gemm_bf16_operands(st, C.byref(g))
    lib.nchip_gemm_bf16_operands_class(0)
    c, p, c16 = hip.numpy(t["c"]), hip.numpy(t["pre"]), hip.numpy(t["c16"])
    hip.free(*t.values())
    if tb and n % 64:
        # a column-contiguous B must fill whole tiles: the entry point declines (1 = "use the
        # route that rounds on the fly") and leaves the outputs alone
        assert rc == 1 and (c == 7.0).all() and (p == 7.0).all() and (c16 == 7).all()
        return
    if rc == 1:                                 # (only the 128-wide class may decline 192 columns)
        assert tb and n % 128 and cls == 1 and (c == 7.0).all()
        return
    assert rc == 0
    assert relerr(p, pre) <= 1e-5
    assert relerr(c, want) <= 1e-5
    assert np.array_equal(c16, bf16_round(c)[1])        # the copy is the rounding of what C holds


def test_activation_gradient_epilogue_and_row_sums(hip, raw, rng):
    lib, st, ptr = raw
    m, n, k = 256, 384, 128                      # dX (m, n) = W^T (m, k) dY (k, n), times gelu'(pre)
    w = rng.standard_normal((m, k)).astype(np.float32)        # column-major (k, m): ta = 1
    dy = rng.standard_normal((n, k)).astype(np.float32)
    pre = rng.standard_normal((n, m)).astype(np.float32)
    want = (bf16_round(dy)[0].astype(np.float64) @ bf16_round(w)[0].astype(np.float64).T) * gelu_grad(pre.astype(np.float64))
    lib.nchip_gemm_rowsum_rows.restype = C.c_int
    rows = lib.nchip_gemm_rowsum_rows(n)
    t = dict(w=hip.tensor(w), dy=hip.tensor(dy), pre=hip.tensor(pre), w16=hip.tensor(np.zeros(w.shape, np.uint16)),
             dy16=hip.tensor(np.zeros(dy.shape, np.uint16)), c=hip.tensor(np.zeros((n, m), np.float32)),
             c16=hip.tensor(np.zeros((n, m), np.uint16)), rs=hip.tensor(np.full((rows, m), 9.0, np.float32)))
    lib.nchip_cast_bf16(st, ptr(t["w"]), ptr(t["w16"]), w.size)
    lib.nchip_cast_bf16(st, ptr(t["dy"]), ptr(t["dy16"]), dy.size)
    written = C.c_int(0)
    g = Args(ta=1, tb=0, m=m, n=n, k=k, alpha=1.0, A16=ptr(t["w16"]), B16=ptr(t["dy16"]), lda=k, ldb=k,
             C=ptr(t["c"]), ldc=m, C16=ptr(t["c16"]), dpre=ptr(t["pre"]), dact=1, rowsum=ptr(t["rs"]),
             rows_written=C.pointer(written))
    assert lib.nchip_gemm_bf16_operands(st, C.byref(g)) == 0
    c, c16, rs = hip.numpy(t["c"]), hip.numpy(t["c16"]), hip.numpy(t["rs"])
    hip.free(*t.values())
    assert relerr(c, want) <= 1e-5
    assert np.array_equal(c16, bf16_round(c)[1])
    assert 0 < written.value <= rows
    assert relerr(rs[: written.value].sum(axis=0), c.astype(np.float64).sum(axis=0)) <= 1e-5


def test_grouped_launch_from_bf16_operands(hip, raw, rng):
    """dW = alpha (dY X^T + dY2 X2^T) for three problems of different sizes in one launch."""
    lib, st, ptr = raw
    probs = [(256, 128, 192, 64), (128, 384, 64, 0), (512, 256, 128, 128)]   # (m, n, k, k2)
    keep, table, wants, outs, tiles, flops = [], [], [], [], 0, 0.0
    for m, n, k, k2 in probs:
        ops = [rng.standard_normal((kk, dim)).astype(np.float32) for kk, dim in ((k, m), (k, n), (k2, m), (k2, n)) if kk]
        dev = [hip.tensor(o) for o in ops]
        d16 = [hip.tensor(np.zeros(o.shape, np.uint16)) for o in ops]
        for s_, d_, o in zip(dev, d16, ops):
            assert lib.nchip_cast_bf16(st, ptr(s_), ptr(d_), o.size) == 0
        r = [bf16_round(o)[0].astype(np.float64) for o in ops]
        want = r[1].T @ r[0] + (r[3].T @ r[2] if k2 else 0.0)                 # (n, m) numpy = column-major (m, n)
        out = hip.tensor(np.full((n, m), 5.0, np.float32))
        table.append(Problem(A=ptr(d16[0]), B=ptr(d16[1]), C=ptr(out), A2=ptr(d16[2]) if k2 else None,
                             B2=ptr(d16[3]) if k2 else None, m=m, n=n, k=k, k2=k2, lda=m, ldb=n, ldc=m,
                             tile_start=tiles, alpha=0.5))
        tiles += (m // 128) * (n // 128)
        flops += 2.0 * m * n * (k + k2)
        wants.append(0.5 * want)
        outs.append(out)
        keep += dev + d16
    raw_table = np.frombuffer(b"".join(bytes(p) for p in table), dtype=np.uint8)
    dev_table = hip.tensor(raw_table)
    assert lib.nchip_gemm_grouped(st, 0, 1, ptr(dev_table), len(table), tiles, 2, flops) == 0
    for out, want in zip(outs, wants):
        assert relerr(hip.numpy(out), want) <= 1e-5
    hip.free(dev_table, *outs, *keep)


def test_tensor_products_in_bf16_mode_use_and_keep_shadows(hip, ref, rng):
    """nc_linear / nc_matmul with bf16 products on: forward, the activation-gradient product,
    the input gradients and the weight gradients of a two-layer perceptron agree with
    the checker's emulation of the same rounding (2e-2 is the variant's bar; these agree to
    fp32 summation error), on shapes that take the shadow route and on shapes that do not;
    an operand rewritten in place between two products is read again, not remembered."""
    for d, f, n in ((128, 256, 192), (128, 256, 50), (96, 200, 64)):
        w1 = (rng.standard_normal((d, f)) * 0.1).astype(np.float32)       # numpy (d, f) = column-major (f, d)
        w2 = (rng.standard_normal((f, d)) * 0.1).astype(np.float32)
        b1 = rng.standard_normal(f).astype(np.float32)
        x = rng.standard_normal((n, d)).astype(np.float32)
        res = []
        for nc in (hip, ref):
            nc.nc_set_matmul_bf16(nc.ctx, 1)
            (h1, p1), (h2, p2), (hb, pb) = nc.param(w1, "w1"), nc.param(w2, "w2"), nc.param(b1, "b1")
            hx, px = nc.param(x, "x")
            y = nc.nc_linear(nc.dup(h1.value), nc.dup(hx.value), nc.dup(hb.value), 1)
            y = nc.nc_matmul(nc.dup(h2.value), y)
            out = nc.numpy(y)
            loss = nc.nc_sum(nc.nc_mul(y, nc.tensor(np.linspace(-1, 1, out.size, dtype=np.float32).reshape(out.shape))))
            grads = nc.backward(loss)
            nc.free(loss)
            res.append((out, [grads[p] for p in (p1, p2, pb, px)]))
            # the same product again after x was rewritten in place: must see the new values
            x2 = x[::-1].copy()
            src = nc.tensor(x2)
            nc.nc_tensor_copy(hx.value, src)
            nc.free(src)
            y2 = nc.nc_matmul(nc.dup(h1.value), nc.dup(hx.value))
            res[-1] = res[-1] + (nc.numpy(y2, free=True),)
            nc.nc_set_matmul_bf16(nc.ctx, 0)
        (o_h, g_h, y2_h), (o_r, g_r, y2_r) = res
        # one product: fp32 summation error.  A chain of two: an activation that sits near a
        # rounding boundary may round to the other bf16 neighbour on the two sides (2^-9 of
        # that element), which is what the looser bars of the chained results allow for.
        assert relerr(y2_h, y2_r) <= 2e-5, (d, f, n)
        assert relerr(o_h, o_r) <= 5e-4, (d, f, n)
        for a, b in zip(g_h, g_r):
            assert relerr(a, b) <= 2e-3, (d, f, n)


def test_training_steps_through_shadows_match_the_checkers_emulation():
    """Three RMSProp steps of a two-layer model whose every product takes the bf16-operand
    route (d_model 128, 128 tokens per segment: forward, input-gradient, activation-gradient
    and the grouped weight-gradient launch), with the shadow checker on: every copy a product
    reads is compared with a fresh rounding of its buffer first (a stale copy ends the
    process).  Probabilities, loss and parameters against the checker emulating the same
    operand rounding, at the variant's bar; memories shift between the steps (mem_len >
    seg_len), so copies of rewritten buffers must be dropped."""
    import modelutil as M
    hp = M.load_pkg().host
    cfg = dict(n_layer=2, d_model=128, n_head=2, d_inner=256, d_pos=48, mem_len=32, seg_len=16,
               batch_size=8, n_symbols=64, seed=11)
    syms = M.markov1(cfg["batch_size"] * cfg["seg_len"] * 3, cfg["n_symbols"], seed=12)
    batches = M.segment_batches(syms, cfg["batch_size"], cfg["seg_len"], 3)
    res = []
    for host, dev in ((M.hip_host(), 1), (M.ref_host(), 0)):
        m = hp.Model(host, hp.make_config(**dict(cfg, use_device=dev, fused=1, nb_threads=4, sgd_opt=M.rmsprop(3e-4))))
        m.nc.nc_set_matmul_bf16(m.ctx, 1)
        old = m.nc.nc_set_bf16_shadow_check(1)
        steps = [m.train_step(tok, tgt, 3e-4) for tok, tgt in batches]
        casts = m.nc.nc_get_bf16_cast_count(m.ctx)
        w = m.params()
        m.nc.nc_set_bf16_shadow_check(old)
        m.nc.nc_set_matmul_bf16(m.ctx, 0)
        m.close()
        res.append((steps, w, casts))
    (s_h, w_h, casts), (s_r, w_r, _) = res
    assert casts > 0                                  # the route was taken (embedding output, attention output, ...)
    for (p_h, l_h), (p_r, l_r) in zip(s_h, s_r):
        assert M.relerr(p_h, p_r) <= 2e-2
        assert abs(l_h - l_r) <= 2e-2 * abs(l_r)
    for k in w_r:
        if w_r[k].ndim >= 2 and not k.startswith("b_r"):
            assert M.rel_l2(w_h[k], w_r[k]) <= 2e-2, k


ATTN_CFGS = [dict(H=2, B=2, T=64, M=64, d_pos=128, attn_len=128),      # the headline head shape
             dict(H=1, B=3, T=48, M=80, d_pos=128, attn_len=100),
             dict(H=2, B=2, T=40, M=24, d_pos=64, attn_len=64),        # key tiles partly empty
             dict(H=2, B=1, T=64, M=64, d_pos=40, attn_len=128),       # far keys share position row 0
             dict(H=1, B=2, T=64, M=192, d_pos=256, attn_len=256),     # 256 keys: the 16-tile instantiation
             dict(H=2, B=2, T=17, M=143, d_pos=160, attn_len=90),
             dict(H=2, B=2, T=64, M=64, d_pos=0, attn_len=128),        # no position vectors
             dict(H=2, B=2, T=33, M=17, d_pos=29, attn_len=25)]        # K not a multiple of 8: the fp32 kernels


@pytest.mark.parametrize("cfg", ATTN_CFGS)
def test_attention_on_the_bf16_matrix_cores(hip, ref, rng, cfg):
    """nc_relpos_attention with bf16 products on: q, kv, kv_mem and w_r are read as bf16, the
    probabilities, dS, dRel and dO are rounded to bf16 where a product multiplies them, sums are
    fp32.  Against the checker's fp32 attention on inputs that are already bf16 values (so the
    operand rounding is exact on both sides): what is left is the rounding of the
    intermediate factors, 2^-9 each - output and every gradient within 1e-2 of their
    largest magnitude, an order inside the variant's 2e-2 bar and an order above what the
    fp32 path holds (1e-5).  The launch count shows which kernels ran."""
    H, B, T, M, d_pos = (cfg[k] for k in ("H", "B", "T", "M", "d_pos"))
    dk = dv = 64
    K = M + T
    shapes = [(T, B, H * dk), (T, B, H * (dk + dv)), (M, B, H * (dk + dv)), (H, max(d_pos, 1), dk), (H, K)]
    arrays = [bf16_round((rng.standard_normal(s) * 0.5).astype(np.float32))[0] for s in shapes]
    weight = bf16_round(rng.standard_normal((T, B, H * dv)).astype(np.float32))[0]
    res = []
    for nc in (hip, ref):
        nc.nc_set_matmul_bf16(nc.ctx, 1)
        old = nc.nc_set_bf16_shadow_check(1)
        hs = [nc.param(a, "p%d" % i) for i, a in enumerate(arrays)]
        args = [nc.dup(h.value) for h, _ in hs]
        if d_pos == 0:
            nc.free(args[3])
            args[3] = None
        l0 = nc.nc_get_launch_count(nc.ctx)
        y = nc.nc_relpos_attention(*args, H, dk, cfg["attn_len"], 2.5)
        fwd_launches = nc.nc_get_launch_count(nc.ctx) - l0
        out = nc.numpy(y)
        loss = nc.nc_sum(nc.nc_mul(y, nc.tensor(weight)))
        g = nc.backward(loss)
        nc.free(loss)
        res.append((out, [g.get(p) for _, p in hs], fwd_launches))
        nc.nc_set_bf16_shadow_check(old)
        nc.nc_set_matmul_bf16(nc.ctx, 0)
    (o_h, g_h, launches), (o_r, g_r, _) = res
    assert relerr(o_h, o_r) <= 1e-2
    for i, (a, b) in enumerate(zip(g_h, g_r)):
        if d_pos == 0 and i == 3:
            continue
        assert relerr(a, b) <= 1e-2, i
    if K % 8 == 0:
        assert launches <= 5            # 4 casts at most (parameters here have no producer) + the one kernel


@pytest.mark.parametrize("ta,tb,m,n,k,pad", [(0, 0, 320, 70, 64, 0), (1, 0, 75, 131, 128, 1), (0, 1, 192, 128, 192, 2),
                                             (1, 1, 130, 64, 320, 3), (1, 0, 260, 257, 576, 0), (0, 1, 64, 320, 448, 4)])
def test_tile_classes_give_the_same_bits_at_the_edges_of_tiles_and_stages(hip, raw, rng, ta, tb, m, n, k, pad):
    """Every class, 1 to 9 stages of 64 k, partial tiles in both directions, columns of C that are not
    16-byte aligned: one chain over k for each element, so every class writes the same C (and a
    copy that is its rounding), within fp32 summation error (k roundings of 2^-24) of float64."""
    lib, st, ptr = raw
    a = rng.standard_normal((m, k) if ta else (k, m)).astype(np.float32)
    b = rng.standard_normal((k, n) if tb else (n, k)).astype(np.float32)
    ra, rb = bf16_round(a), bf16_round(b)
    am, bm = (ra[0] if not ta else ra[0].T).astype(np.float64), (rb[0] if not tb else rb[0].T).astype(np.float64)
    pre, add, bias = (rng.standard_normal(s).astype(np.float32) for s in ((n, m + pad), (n, m + pad), (m,)))
    product, scale = bm @ am, np.abs(bm) @ np.abs(am)
    lib.nchip_gemm_rowsum_rows.restype = C.c_int
    rows = lib.nchip_gemm_rowsum_rows(n)
    first = {}
    for cls in (1, 2, 3, 4, 5):
        for mode in ("forward", "backward"):
            t = dict(a=hip.tensor(ra[1]), b=hip.tensor(rb[1]), pre=hip.tensor(pre), add=hip.tensor(add), bias=hip.tensor(bias),
                     c=hip.tensor(np.full((n, m + pad), 7.0, np.float32)), c16=hip.tensor(np.full((n, m + pad), 7, np.uint16)),
                     rs=hip.tensor(np.zeros((rows, m), np.float32)))
            written = C.c_int(0)
            g = Args(ta=ta, tb=tb, m=m, n=n, k=k, alpha=1.0, A16=ptr(t["a"]), B16=ptr(t["b"]), lda=k if ta else m,
                     ldb=n if tb else k, C=ptr(t["c"]), ldc=m + pad, C16=ptr(t["c16"]))
            if mode == "forward":
                g.bias, g.act, g.addend, want = ptr(t["bias"]), 2, ptr(t["add"]), np.maximum(product + bias, 0) + add[:, :m]
            else:
                g.dpre, g.dact, g.rowsum, g.rows_written = ptr(t["pre"]), 2, ptr(t["rs"]), C.pointer(written)
                want = product * (pre[:, :m] > 0)
            lib.nchip_gemm_bf16_operands_class(cls)
            assert lib.nchip_gemm_bf16_operands(st, C.byref(g)) == 0
            lib.nchip_gemm_bf16_operands_class(0)
            c, c16, rs = hip.numpy(t["c"]), hip.numpy(t["c16"]), hip.numpy(t["rs"])
            hip.free(*t.values())
            assert np.all(np.abs(c[:, :m] - want) <= 2.0 ** -24 * (k + 2) * (scale + np.abs(bias) + np.abs(add[:, :m])))
            assert (c[:, m:] == 7.0).all() and (c16[:, m:] == 7).all() and np.array_equal(c16[:, :m], bf16_round(c[:, :m])[1])
            assert np.array_equal(first.setdefault(mode, c), c)
            if mode == "backward":  # 16 columns a partial row, added in some order
                bound = 2.0 ** -24 * 16 * np.abs(c[:, :m]).astype(np.float64).sum(0)
                assert np.all(np.abs(rs[: written.value].astype(np.float64).sum(0) - c[:, :m].astype(np.float64).sum(0)) <= bound)


def test_grouped_launch_in_wide_tiles(hip, raw, rng):
    """nchip_gemm_grouped with precision 3: problems of 128 rows or columns inside 256-wide tiles, one of
    two k ranges; the bits of the 128-wide launch."""
    lib, st, ptr = raw
    tables = {2: [], 3: []}
    keep, outs, tiles = [], {2: [], 3: []}, {2: 0, 3: 0}
    for m, n, k, k2 in [(384, 128, 192, 64), (128, 512, 64, 0), (256, 256, 128, 128)]:
        d = [hip.tensor(bf16_round(rng.standard_normal((kk, dim)).astype(np.float32))[1])
             for kk, dim in ((k, m), (k, n), (k2, m), (k2, n)) if kk]
        keep += d
        for prec, tile, count in ((2, 128, lib.nchip_gemm_grouped_tiles), (3, 256, lib.nchip_gemm_grouped_tiles256)):
            out = hip.tensor(np.full((n, m), 5.0, np.float32))
            tables[prec].append(Problem(A=ptr(d[0]), B=ptr(d[1]), C=ptr(out), A2=ptr(d[2]) if k2 else None,
                                        B2=ptr(d[3]) if k2 else None, m=m, n=n, k=k, k2=k2, lda=m, ldb=n, ldc=m,
                                        tile_start=tiles[prec], alpha=0.5))
            tiles[prec] += -(-m // tile) * -(-n // tile)
            assert count(m, n) == -(-m // tile) * -(-n // tile)
            outs[prec].append(out)
    for prec in (2, 3):
        table = hip.tensor(np.frombuffer(b"".join(bytes(p) for p in tables[prec]), dtype=np.uint8))
        assert lib.nchip_gemm_grouped(st, 0, 1, ptr(table), len(tables[prec]), tiles[prec], prec, 1.0) == 0
        keep.append(table)
    for two, three in zip(outs[2], outs[3]):
        assert np.array_equal(hip.numpy(two), hip.numpy(three))
    hip.free(*keep, *outs[2], *outs[3])


def _precision_1(lib, st, ptr, ta, tb, m, n, k, a_t, b_t, c_t):
    p, i, j, f = C.c_void_p, C.c_int, C.c_int64, C.c_float
    lib.nchip_gemm.argtypes = [p, i, i, i, i, i, f, p, j, j, p, j, j, f, p, j, j, i, p, i, p, i, i, p]
    return lib.nchip_gemm(st, ta, tb, m, n, k, 1.0, ptr(a_t), k if ta else m, 0, ptr(b_t), n if tb else k, 0, 0.0, ptr(c_t), m, 0, 1,
                          None, 0, None, 1, 1, None)


@pytest.mark.parametrize("ta,tb,m,n,k", [(0, 0, 100, 67, 64), (1, 0, 130, 131, 200), (0, 1, 257, 96, 352), (1, 1, 65, 300, 129), (0, 1, 128, 256, 1024)])
def test_products_from_rounded_copies_keep_two_chains_below_512_tiles(hip, raw, rng, ta, tb, m, n, k):
    """nchip_gemm with precision 1 through rounded copies: the bits of the tile loader's rounding in the 64x64
    class, which gives an element two chains over k, and with one chain forced those of the 128x128 class."""
    lib, st, ptr = raw
    a_t, b_t = (hip.tensor(rng.standard_normal(s).astype(np.float32)) for s in ((m, k) if ta else (k, m), (k, n) if tb else (n, k)))
    got = []
    for source, config in ((2, 0), (0, 10), (2, 11), (2, 13), (0, 7)):
        c_t = hip.tensor(np.full((n, m), 7.0, np.float32))
        lib.nchip_gemm_bf16_source(source)
        lib.nchip_gemm_force_config(config)
        rc = _precision_1(lib, st, ptr, ta, tb, m, n, k, a_t, b_t, c_t)
        lib.nchip_gemm_force_config(0)
        lib.nchip_gemm_bf16_source(1)
        assert rc == 0
        got.append(hip.numpy(c_t, free=True))
    hip.free(a_t, b_t)
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[2], got[1])
    assert np.array_equal(got[3], got[4])
    assert not np.array_equal(got[0], got[3])


@pytest.mark.parametrize("ta,tb,m,n,k", [(0, 0, 192, 7110, 64), (0, 0, 192, 8200, 64), (1, 1, 130, 14272, 64)])
def test_bf16_operands_that_do_not_fill_their_tiles_have_the_sums_of_the_general_call(hip, raw, rng, ta, tb, m, n, k):
    """192 rows in 128-wide tiles, columns that are a multiple of 64 and not of 128: the bits of nchip_gemm with
    precision 1, whose class for the shape has one chain over k or two."""
    lib, st, ptr = raw
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((m, k) if ta else (k, m), (k, n) if tb else (n, k)))
    a_t, b_t, c_t, d_t, a16, b16 = (hip.tensor(x) for x in (a, b, np.full((n, m), 7.0, np.float32), np.full((n, m), 8.0, np.float32),
                                                             bf16_round(a)[1], bf16_round(b)[1]))
    assert _precision_1(lib, st, ptr, ta, tb, m, n, k, a_t, b_t, c_t) == 0
    g = Args(ta=ta, tb=tb, m=m, n=n, k=k, alpha=1.0, A16=ptr(a16), B16=ptr(b16), lda=k if ta else m, ldb=n if tb else k, C=ptr(d_t), ldc=m)
    assert lib.nchip_gemm_bf16_operands(st, C.byref(g)) == 0
    assert np.array_equal(hip.numpy(c_t), hip.numpy(d_t))
    hip.free(a_t, b_t, c_t, d_t, a16, b16)


@pytest.mark.parametrize("far,m,n,k,ld", [("a", 3, 70, 128, (1 << 30) + 8), ("b", 66, 64, 64, (1 << 25) + (1 << 21))])
def test_bf16_operands_with_rows_gigabytes_apart(hip, raw, rng, far, m, n, k, ld):
    """Rows whose offsets inside a stage pass 32 bits (k contiguous, and n contiguous): the bits of the compact
    operands.  One operand lies in a buffer of 4.3 GB, of which only its rows are written."""
    lib, st, ptr = raw
    tb = far == "b"
    rows = {"a": rng.standard_normal((m, k)).astype(np.float32), "b": rng.standard_normal((k, n) if tb else (n, k)).astype(np.float32)}
    one = {"a": k, "b": n if tb else k}
    n_big = (len(rows[far]) - 1) * ld + one[far]
    big = hip.lib.nc_new_tensor_nz(hip.dev, 0, 1, (C.c_size_t * 1)((n_big + 1) // 2))  # (f32: two values each)
    d = {x: hip.tensor(r) for x, r in rows.items()}
    d16 = {x: hip.tensor(np.zeros(r.shape, np.uint16)) for x, r in rows.items()}
    for x, r in rows.items():
        assert lib.nchip_cast_bf16(st, ptr(d[x]), ptr(d16[x]), r.size) == 0
    for i in range(len(rows[far])):
        assert lib.nchip_cast_bf16(st, C.c_void_p(ptr(d[far]).value + 4 * i * one[far]), C.c_void_p(ptr(big).value + 2 * i * ld), one[far]) == 0
    got = []
    for a16, lda, b16, ldb in ((d16["a"], one["a"], d16["b"], one["b"]), (big if far == "a" else d16["a"], ld if far == "a" else one["a"],
                                                                          big if far == "b" else d16["b"], ld if far == "b" else one["b"])):
        c_t = hip.tensor(np.full((n, m), 7.0, np.float32))
        g = Args(ta=1, tb=int(tb), m=m, n=n, k=k, alpha=1.0, A16=ptr(a16), B16=ptr(b16), lda=lda, ldb=ldb, C=ptr(c_t), ldc=m)
        assert lib.nchip_gemm_bf16_operands(st, C.byref(g)) == 0
        got.append(hip.numpy(c_t, free=True))
    hip.free(big, *d.values(), *d16.values())
    assert np.array_equal(*got)


def _grouped_products(hip, raw, problems, precision, tiles_of, ta, tb, start=0.0):
    """C of each (a, b, a2, b2) - stored (columns, rows), a2 / b2 or None - through one grouped launch."""
    lib, st, ptr = raw
    keep, outs, table, tiles = [], [], b"", 0
    for a, b, a2, b2 in problems:
        (k, m), (n, kb) = (a.shape if not ta else a.shape[::-1]), (b.shape if not tb else b.shape[::-1])
        assert k == kb
        d = [None if x is None else hip.tensor(x) for x in (a, b, a2, b2)]
        out = hip.tensor(np.full((n, m), start, np.float32))
        k2 = 0 if a2 is None else a2.shape[1 if ta else 0]
        table += bytes(Problem(A=ptr(d[0]), B=ptr(d[1]), C=ptr(out), A2=ptr(d[2]) if k2 else None, B2=ptr(d[3]) if k2 else None,
                               m=m, n=n, k=k, k2=k2, lda=k if ta else m, ldb=n if tb else k, ldc=m, tile_start=tiles, alpha=0.5))
        tiles += tiles_of(m, n)
        keep += [x for x in d if x]
        outs.append(out)
    t = hip.tensor(np.frombuffer(table, dtype=np.uint8))
    assert lib.nchip_gemm_grouped(st, ta, tb, ptr(t), len(problems), tiles, precision, 1.0) == 0
    got = [hip.numpy(x, free=True) for x in outs]
    hip.free(t, *keep)
    return got


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_grouped_fp32_launch_by_whole_units(hip, raw, rng, ta, tb):
    """nchip_gemm_grouped with precision 4: partial tiles, ranges of one stage and of several, a second range (with k
    contiguous in neither operand: the two share their leading dimensions), no k at all: the bits of precision 0."""
    def operands(m, n, k):
        return (rng.standard_normal((m, k) if ta else (k, m)).astype(np.float32), rng.standard_normal((k, n) if tb else (n, k)).astype(np.float32))
    problems = []
    for m, n, k, k2 in [(4, 132, 32, 32), (260, 64, 160, 32), (128, 128, 96, 288), (68, 4, 256, 0), (32, 36, 0, 0)]:
        second = operands(m, n, k2) if k2 and not ta and tb else (None, None)
        problems.append(operands(m, n, k) + second if k else (np.zeros((m, 0) if ta else (0, m), np.float32), np.zeros((0, n) if tb else (n, 0), np.float32), None, None))
    lib = raw[0]
    zero, four = (_grouped_products(hip, raw, problems, p, lib.nchip_gemm_grouped_tiles, ta, tb, 5.0) for p in (0, 4))
    assert all(np.array_equal(x, y) for x, y in zip(zero, four)) and not four[-1].any()


@pytest.mark.parametrize("precision", [0, 1, 5, 6])
def test_grouped_launch_of_any_k(hip, raw, rng, precision):
    """Ranges that end inside a stage, and the launch that adds to what C holds: float64 of the same operands (bf16
    values, so that both precisions form the same products) within a rounding per addition."""
    bf = lambda *s: bf16_round(rng.standard_normal(s).astype(np.float32))[0]
    shapes = [(37, 70, 5, 33), (130, 64, 131, 97), (129, 257, 64, 1), (5, 3, 1, 0)]
    problems = [(bf(k, m), bf(k, n), bf(k2, m) if k2 and precision < 5 else None, bf(k2, n) if k2 and precision < 5 else None) for m, n, k, k2 in shapes]
    lib, start = raw[0], 3.0 if precision >= 5 else 0.0
    got = _grouped_products(hip, raw, problems, precision, lib.nchip_gemm_grouped_tiles64 if precision >= 5 else lib.nchip_gemm_grouped_tiles, 0, 1, 3.0)
    for (a, b, a2, b2), c in zip(problems, got):
        a, b = (np.concatenate([x] if y is None else [x, y]).astype(np.float64) for x, y in ((a, a2), (b, b2)))
        assert np.all(np.abs(c - (0.5 * b.T @ a + start)) <= 2.0 ** -24 * (len(a) + 2) * (np.abs(b).T @ np.abs(a) + start))
