"""Kernels at the sizes where they can go wrong - tile edges, remainders, the smallest and
largest of a range - against the CPU checker or a float64 statement."""
import ctypes as C

import numpy as np
import pytest

import cases
import modelutil as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 255, 257, 16384, 16385, 65537, 300001, (1 << 20) + 77])
def test_random_fill_across_runs_and_wavefronts(hip, ref, n):
    """A fill starts every run of 256 elements and every wavefront of 64 runs from a state it
    jumps to: each element, and the state the fill leaves behind (seen by the next one), is the
    serial stream's."""
    got = []
    for nc in (hip, ref):
        rs = nc.lib.nc_rnd_init(nc.dev, 77)
        one = []
        for size in (n, 5, n):
            t = nc.tensor(np.zeros(size, np.float32))
            nc.lib.nc_tensor_set_rnd_unif(t, 0.5, 0.25, rs)
            one.append(nc.numpy(t, free=True))
            t = nc.tensor(np.zeros(size, np.float32))
            nc.lib.nc_tensor_set_dropout(t, 0.19, rs)
            one.append(nc.numpy(t, free=True))
        nc.lib.nc_rnd_end(rs)
        got.append(one)
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_random_fill_takes_every_jump(hip, ref):
    """8193 wavefronts and a bit: the start state of one is a product over the bits of its index, so
    all fourteen jump matrices are taken, each alone and with others."""
    n, got = (1 << 27) + 16384 + 5, []
    for nc in (hip, ref):
        rs = nc.lib.nc_rnd_init(nc.dev, 77)
        t = nc.nc_new_tensor_nz(nc.dev, 0, 1, (C.c_size_t * 1)(n))
        nc.lib.nc_tensor_set_rnd_unif(t, 0.5, 0.25, rs)
        got.append(nc.numpy(t, free=True).view(np.uint32))
        nc.lib.nc_rnd_end(rs)
    assert np.array_equal(*got)


@pytest.mark.parametrize("first,last", [(0, 40), (1, 40), (3, 4), (8, 33), (37, 40)])
def test_random_fill_of_a_bf16_range(hip, ref, first, last):
    """A range of a bf16 tensor at any start: the checker's bits, and its neighbours untouched."""
    got = []
    for nc in (hip, ref):
        rs = nc.lib.nc_rnd_init(nc.dev, 5)
        t = nc.nc_convert(nc.tensor(np.full(40, 2.0, np.float32)), 1)
        a = nc.nc_slice_alias(t, 0, first, last)
        nc.lib.nc_tensor_set_rnd_unif(a, 0.5, 0.25, rs)
        nc.free(a)
        got.append(nc.numpy(t, free=True))
        nc.lib.nc_rnd_end(rs)
    assert np.array_equal(*got)


@pytest.mark.parametrize("shape", [(2, 3, 5, 8), (2, 3, 5, 7), (3, 1, 4, 4), (1, 1, 1, 1), (7, 2, 33, 12)])
def test_permuted_copies_and_broadcasts(hip, shape):
    """Leading axes of whole 16-byte units and others, through the strided copy (a head split and
    its inverse) and the broadcast sums and products: exact copies, exact float32 results."""
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal(shape).astype(np.float32)            # libnc dims are the reverse
    y = hip.nc_permute_4d(hip.tensor(x), 0, 3, 1, 2)             # axis a of the result is axis p[a] of x
    assert np.array_equal(hip.numpy(y, free=True), np.transpose(x, (1, 2, 0, 3)))
    for b in (x[0, 0, 0], x[0, 0], x[0, 0, 0, :1].reshape(())):  # a prefix of the axes, and a scalar
        a = hip.numpy(hip.nc_add(hip.tensor(x), hip.tensor(b)), free=True)
        m = hip.numpy(hip.nc_mul(hip.tensor(x), hip.tensor(b)), free=True)
        assert np.array_equal(a, x + b) and np.array_equal(m, x * b)


@pytest.mark.parametrize("n,first,last", [(1, 0, 1), (17, 1, 16), (40, 3, 37), (4096, 0, 4096), (100003, 5, 99998)])
def test_zeroed_ranges_keep_their_neighbours(hip, n, first, last):
    x = np.arange(1, n + 1, dtype=np.float32)
    t = hip.tensor(x)
    a = hip.nc_slice_alias(t, 0, first, last)
    hip.nc_tensor_set_zero(a)
    hip.free(a)
    x[first:last] = 0
    assert np.array_equal(hip.numpy(t, free=True), x)


@pytest.fixture(scope="module")
def hosts():
    return M.hip_host(), M.ref_host()


@pytest.mark.parametrize("cells,batch,seg,variant", [
    (1, 1, 1, dict()), (15, 3, 2, dict(lstm_type=2)), (17, 33, 3, dict(lstm_type=0, lstm_use_layer_norm=0)),
    (64, 16, 4, dict(lstm_full_connect=0)), (257, 5, 3, dict()), (385, 2, 2, dict(lstm_type=2, lstm_use_layer_norm=0)),
    (520, 1, 2, dict(n_layer=1))])
def test_lstm_layer_sizes(hosts, cells, batch, seg, variant):
    """The per-layer kernels against the checker's op-by-op sequence: units around 256 and 512 (one,
    two and four per thread), tiles of 16 with remainders, unaligned columns, three and four gates,
    with and without the norm.  Bar: the single-step 1e-5 of the model tests, on probabilities,
    loss and, through one step of plain SGD, every gradient; a gain's gradient, one number that sums
    terms of both signs over all units and columns, to 2^-24 sqrt(terms) of its largest terms: 1e-4."""
    pkg = M.load_pkg()
    cfg = dict(n_layer=2, lstm_n_cells=cells, batch_size=batch, seg_len=seg, n_symbols=31, seed=5, sgd_opt=M.sgd(0.5))
    cfg.update(variant)
    hip = pkg.host.Model(hosts[0], pkg.host.make_lstm_config(**dict(cfg, use_device=1)))
    ref = pkg.host.Model(hosts[1], pkg.host.make_lstm_config(**dict(cfg, use_device=0, nb_threads=4)))
    syms = M.markov1(batch * seg * 2, 31, seed=7)
    for tok, tgt in M.segment_batches(syms, batch, seg, 2):      # the second from a carried state
        ph, lh = hip.train_step(tok, tgt, 0.5)
        pr, lr = ref.train_step(tok, tgt, 0.5)
        assert M.relerr(ph, pr) <= 1e-5 and abs(lh - lr) <= 1e-5 * abs(lr)
    w_h, w_r = hip.params(), ref.params()
    for k in w_r:
        assert M.rel_l2(w_h[k], w_r[k]) <= (1e-4 if w_r[k].size == 1 else 1e-5), (k, M.rel_l2(w_h[k], w_r[k]))
    hip.close()
    ref.close()


@pytest.mark.parametrize("cells,batch,seg,variant", [
    (33, 5, 6, dict()), (130, 17, 5, dict(lstm_type=0, lstm_use_layer_norm=0)), (70, 9, 8, dict(lstm_type=2))])
def test_lstm_layer_against_float64(hosts, cells, batch, seg, variant):
    """The per-layer kernels sum in another order than the sequence of ops: whether that loses
    accuracy is decided by a float64 evaluation of the segment.  Probabilities and every gradient (exposed by
    one step of plain SGD at a rate that lifts it above the weights, w0 - w1 = 2^20 g) are no further
    from it than twice what the checker's sequence is, each kind of tensor taken together (a gain's
    gradient is one number, the sum of many terms of both signs).  Measured, per layer against
    sequence: probabilities 0.9-1.3e-7 against
    1.2-1.8e-7, recurrent weights 1.8-2.4e-7 against 1.9-2.9e-7, biases 1.4-2.0e-7 against
    1.4-2.7e-7, gains 1.8-2.3e-7 against 2.4-2.5e-7."""
    import torch
    from test_lstm_torch import lstm_forward_torch
    H, lr = M.load_pkg().host, float(1 << 20)
    cfg = dict(n_layer=2, lstm_n_cells=cells, batch_size=batch, seg_len=seg, n_symbols=31, seed=5)
    cfg.update(variant)
    rng = np.random.default_rng(cells)
    tok, tgt = rng.integers(0, 31, size=(2, seg, batch)).astype(np.int32)
    got = []
    for host, dev in zip(hosts, (1, 0)):
        m = H.Model(host, H.make_lstm_config(**dict(cfg, use_device=dev, nb_threads=4, sgd_opt=M.sgd(lr))))
        noise = np.random.default_rng(1)
        for k in m.param_names():                    # biases and gains away from their initial 0 / 1
            if k[0] in "bg" or k == "fc_b":
                m.set_param(k, m.get_param(k) + 0.3 * noise.standard_normal(m.get_param(k).shape).astype(np.float32))
        w0 = m.params()
        p, _ = m.train_step(tok, tgt, lr)
        w1 = m.params()
        got.append((p, {k: (w0[k].astype(np.float64) - w1[k]) / lr for k in w0}))
        m.close()
    w = {k: torch.tensor(v.astype(np.float64), requires_grad=True) for k, v in w0.items()}
    logp, _, _ = lstm_forward_torch(w, tok, cfg)
    (-logp.gather(2, torch.as_tensor(tgt, dtype=torch.long).unsqueeze(2)).mean()).backward()
    want = logp.exp().detach().numpy()
    kinds = {"probabilities": (got[0][0], got[1][0], want)}
    for kind in ("u", "w", "ws", "b", "g", "fc_w", "fc_b"):
        names = [k for k in w if k.rstrip("_0123456789") == kind]
        if names:
            kinds[kind] = [np.concatenate([np.ravel(t[k]) for k in names])
                           for t in (got[0][1], got[1][1], {k: w[k].grad.numpy() for k in names})]
    errors = {k: (M.rel_l2(a, x), M.rel_l2(b, x)) for k, (a, b, x) in kinds.items()}
    print(" ".join("%s %.1e/%.1e" % (k, *e) for k, e in errors.items()))
    assert len(errors) >= 7 and all(a <= 2.0 * b for a, b in errors.values()), errors


@pytest.mark.parametrize("refused", ["bf16 products", "width invariant", "projection"])
def test_lstm_segment_without_the_layer_form_issues_no_more_than_its_timesteps(hosts, refused):
    """A configuration that has no per-layer form goes straight to the sequence of ops: for segments of
    one timestep the evaluation of the whole segment and that of timestep 0 are one sequence, and
    issue the same launches."""
    H = M.load_pkg().host
    m = H.Model(hosts[0], H.make_lstm_config(n_layer=2, lstm_n_cells=24, lstm_n_cells2=40 if refused == "projection" else 24,
                                             batch_size=3, seg_len=1, n_symbols=31, use_device=1))
    if refused == "bf16 products":
        m.nc.nc_set_matmul_bf16(m.ctx, 1)
    if refused == "width invariant":
        m.nc.nc_set_matmul_width_invariant(m.ctx, 1)
    count = []
    for index in (-1, 0, -1, 0):
        before = m.nc.nc_get_launch_count(m.ctx)
        m.eval(np.zeros((1, 3), np.int32), output_index=index)
        count.append(m.nc.nc_get_launch_count(m.ctx) - before)
    m.close()
    assert count[2] == count[3] > 0, count


@pytest.mark.parametrize("streams,steps", [(65535 * 16 + 1, 1), (1, (1 << 24) + 1)])
def test_lstm_layer_refuses_what_its_launches_cannot_hold(hip, streams, steps):
    """More streams than a grid has rows for, more columns than its indices are laid out for: NULL,
    with nothing consumed or written, and the caller issues the sequence of ops."""
    def dev(*shape):                       # (column-major sizes)
        return hip.nc_new_tensor(hip.dev, 0, len(shape), (C.c_size_t * 8)(*shape))
    pre, u, h, c = dev(3, streams * steps), dev(3, 1), dev(1, streams), dev(1, streams)
    b = (C.c_void_p * 3)(*[dev(1) for _ in range(3)])
    assert not hip.nc_lstm_layer(pre, u, None, b, 3, 2, 1e-5, h, c)
    hip.nc_synchronize(hip.dev)
    hip.free(pre, u, h, c, *b)


@pytest.mark.parametrize("m,n,k,batch", [(1, 1, 1, 1), (16, 16, 16, 1), (17, 15, 63, 3), (33, 7, 64, 2), (31, 5, 65, 1), (40, 20, 256, 2),
                                         (18, 33, 257, 1), (48, 9, 512, 1), (50, 3, 777, 1), (16, 83, 2048, 1), (352, 481, 352, 1), (20, 18, 3072, 1), (20, 18, 3073, 1)])
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
def test_small_products(hip, m, n, k, batch, ta, tb):
    """The 16 x 16 tiles at their edges and at every length of a reduction's round trip, aligned
    columns and others, and the first length past them; the bound is that of a sum of k rounded products in any order."""
    rng = np.random.default_rng(m + 7 * n + k)
    a = rng.standard_normal((batch, m, k)).astype(np.float32)
    b = rng.standard_normal((batch, k, n)).astype(np.float32)
    add = rng.standard_normal((batch, m, n)).astype(np.float32)
    lay = lambda x, t: np.ascontiguousarray(x if t else np.swapaxes(x, 1, 2))  # column major: the first axis last
    got = hip.numpy(hip.nc_matmul_add(hip.tensor(lay(a, ta)), hip.tensor(lay(b, tb)), hip.tensor(lay(add, 0)), ta, tb, 0.5), free=True)
    a, b = a.astype(np.float64), b.astype(np.float64)
    want = 0.5 * (a @ b) + add
    bound = 2.0 ** -24 * ((k + 2) * 0.5 * (np.abs(a) @ np.abs(b)) + 2 * np.abs(add) + np.abs(want))
    assert np.all(np.abs(np.swapaxes(got, 1, 2) - want) <= bound)


def _small_products(hip, m, n, k, batch, ta, tb, pads, options):
    """[small kernel, 64x64 class] results of the products; options: alpha, beta, act, bias, addend"""
    lib = C.CDLL(hip.lib._name)
    rng = np.random.default_rng(m + 7 * n + k)
    st, ci, i64, f32 = C.c_void_p(hip.nc_context_stream(hip.ctx)), C.c_int, C.c_int64, C.c_float
    ks = lib.nchip_gemm_pick_ksplit(ci(m), ci(n), ci(k), ci(batch))
    assert lib.nchip_gemm_is_small(ci(m), ci(n), ci(k), ci(batch)) == 1
    (ra, ca), (rb, cb) = (k, m) if ta else (m, k), (n, k) if tb else (k, n)
    tensors = []

    def dev(x):
        tensors.append(hip.tensor(x.astype(np.float32)))
        return C.c_void_p(hip.nc_tensor_get_ptr(tensors[-1], None))

    bias, ws = dev(rng.standard_normal(m)), dev(np.zeros(batch * ks * m * n))
    try:
        for pad in pads:
            A, B = dev(rng.standard_normal((batch, ca, ra + pad))), dev(rng.standard_normal((batch, cb, rb + pad)))
            add, c0 = rng.standard_normal((2, batch, n, m + pad))
            addp = dev(add)
            for alpha, beta, act, with_bias, with_add in options:
                got = []
                for cfg in (0, 10):
                    lib.nchip_gemm_force_config(cfg)
                    out, pre = dev(c0), dev(np.zeros_like(c0))
                    head = [st, ci(ta), ci(tb), ci(m), ci(n), ci(k), f32(alpha), A, i64(ra + pad), i64(ca * (ra + pad)),
                            B, i64(rb + pad), i64(cb * (rb + pad))]
                    tail = [ci(0), ci(ks), ws]
                    if with_add:
                        rc = lib.nchip_gemm_add(*head, out, i64(m + pad), i64(n * (m + pad)), ci(batch), bias if with_bias else None,
                                                ci(act), pre, addp, *tail)
                    else:
                        rc = lib.nchip_gemm(*head, f32(beta), out, i64(m + pad), i64(n * (m + pad)), ci(batch),
                                            bias if with_bias else None, ci(act), pre, *tail)
                    assert rc == 0
                    got.append([hip.numpy(t) for t in tensors[-2:]])
                yield (k, pad, alpha, beta, act, with_bias, with_add), got
    finally:
        lib.nchip_gemm_force_config(0)
        hip.free(*tensors)


@pytest.mark.parametrize("m,n,k,batch", [(1, 1, 1, 1), (16, 16, 16, 1), (17, 15, 63, 3), (33, 7, 65, 2), (40, 20, 256, 2), (17, 33, 516, 1),
                                         (50, 3, 777, 1), (33, 17, 1023, 1), (33, 17, 1024, 1), (16, 33, 2048, 1), (33, 5, 1500, 2),
                                         (20, 18, 3070, 1)])
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
def test_small_products_have_the_bits_of_their_tile_class(hip, m, n, k, batch, ta, tb):
    """The kernel of 16 x 16 tiles issues the sums of the 64x64 class that the shape would otherwise
    take, split over k or not: the same bits, with every epilogue option of an unforced product,
    from tight columns and from padded ones."""
    options = [(1.0, 0.0, 0, 0, 0), (0.5, 0.0, 0, 0, 1), (1.0, 0.0, 1, 1, 0), (0.5, 0.0, 2, 1, 1), (1.0, 1.0, 0, 0, 0), (0.3, 0.7, 0, 1, 0)]
    for case, (small, tile) in list(_small_products(hip, m, n, k, batch, ta, tb, (0,), options)) + \
            list(_small_products(hip, m, n, k, batch, ta, tb, (1, 4), options[3:4])):
        for u, v in zip(small, tile):
            assert np.array_equal(u, v), (case, np.abs(u - v).max())


@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
def test_small_products_at_every_remainder_of_k(hip, ta, tb):
    """Every remainder of 16 and 32 k behind each number of blocks that a round trip covers (64, 128,
    256, 384 and 512 k)."""
    for k in [*range(1, 34), *range(61, 82), *range(125, 146, 3), *range(255, 290, 2), *range(383, 403, 3), *range(511, 530)]:
        for case, (small, tile) in _small_products(hip, 16, 3, k, 1, ta, tb, (0,), [(1.0, 0.0, 0, 0, 0)]):
            assert np.array_equal(small[0], tile[0]), (case, np.abs(small[0] - tile[0]).max())


def test_a_split_product_without_a_workspace_is_refused(hip):
    """Whatever kernel the shape would go to: -1, and nothing written."""
    lib = C.CDLL(hip.lib._name)
    t = [hip.tensor(np.full((64, 64), 2.0, np.float32)) for _ in range(3)]
    a, b, c = (C.c_void_p(hip.nc_tensor_get_ptr(x, None)) for x in t)
    for k, n in ((64, 8), (16, 64)):
        assert lib.nchip_gemm(C.c_void_p(hip.nc_context_stream(hip.ctx)), 0, 0, 8, n, k, C.c_float(1), a, C.c_int64(64), C.c_int64(0),
                              b, C.c_int64(64), C.c_int64(0), C.c_float(0), c, C.c_int64(64), C.c_int64(0), 1,
                              None, 0, None, 0, 2, None) == -1
    assert np.all(hip.numpy(t[2]) == 2.0)
    hip.free(*t)


@pytest.mark.parametrize("n,h", [(1, 1), (3, 4), (5, 7), (513, 12), (2048, 96)])
@pytest.mark.parametrize("bf16", [0, 1])
def test_geglu_is_its_sequence(hip, n, h, bf16):
    """The one-pass form against nc_split, nc_gelu and nc_mul: the same operations in the same
    order, so the same bits, and the same product of the result (its bf16 copy in bf16 mode)."""
    rng = np.random.default_rng(n + h)
    x = (2 * rng.standard_normal((n, 2 * h))).astype(np.float32)
    w = rng.standard_normal((n, h)).astype(np.float32)
    a = rng.standard_normal((h, 64)).astype(np.float32)
    got = []
    hip.nc_set_matmul_bf16(hip.ctx, bf16)
    try:
        for build in (lambda nc, t: nc.nc_gelu_gate(t), cases._split_build):
            got.append(cases.Case("geglu", [x.shape], build, None).run(hip, [x], w))
            y = build(hip, hip.tensor(x))
            got[-1] += (hip.numpy(hip.nc_matmul(hip.tensor(a), y), free=True),)
    finally:
        hip.nc_set_matmul_bf16(hip.ctx, 0)
    for p, q in zip(*got):
        for u, v in zip(p, q) if isinstance(p, (list, tuple)) else [(p, q)]:
            assert np.array_equal(u, v)


@pytest.mark.parametrize("inner", [2, 63, 65, 700])
@pytest.mark.parametrize("outer", [1, 3, 4, 31, 32, 33, 255, 256, 257])
def test_sums_over_trailing_axes(hip, inner, outer):
    """One launch up to 32 and 256 rows, two past them; the bound is that of a sum in any order."""
    rng = np.random.default_rng(inner + outer)
    x, y0 = rng.standard_normal((outer, inner)).astype(np.float32), rng.standard_normal(inner).astype(np.float32)
    for add in (None, y0):
        got = hip.numpy(hip.nc_reduce_sum(None if add is None else hip.tensor(add), hip.tensor(x), 1), free=True)
        want = x.astype(np.float64).sum(0) + (0 if add is None else add)
        bound = 2.0 ** -24 * ((outer + 1) * np.abs(x).astype(np.float64).sum(0) + np.abs(y0) + np.abs(want))
        assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("m,k,cols", [(17, 5, 3), (64, 32, 16), (130, 70, 40), (96, 64, 300)])
@pytest.mark.parametrize("ta", [0, 1])
def test_gradients_of_a_parameter_used_three_times(hip, m, k, cols, ta):
    """Weights and biases that several products and sums share: the later gradients are added to what
    the parameter holds in the kernel that makes them.  Also one node whose two arguments are the same
    parameter.  Bound: sums of 3 cols rounded products."""
    rng = np.random.default_rng(m + cols)
    w, b = rng.standard_normal((k, m) if not ta else (m, k)).astype(np.float32), rng.standard_normal(m).astype(np.float32)
    xs = [rng.standard_normal((cols, k)).astype(np.float32) for _ in range(3)]
    gs = [rng.standard_normal((cols, m)).astype(np.float32) for _ in range(3)]
    (hw, pw), (hb, pb) = hip.param(w, "w"), hip.param(b, "b")
    loss = hip.nc_sum(hip.nc_mul(hip.dup(hb.value), hip.dup(hb.value)))
    for x, g in zip(xs, gs):
        y = hip.nc_matmul_add(hip.dup(hw.value), hip.tensor(x), None, ta, 0, 1.0)
        y = hip.nc_add(y, hip.dup(hb.value))
        loss = hip.nc_add(loss, hip.nc_sum(hip.nc_mul(y, hip.tensor(g))))
    grads = hip.backward(loss)
    hip.free(loss)
    f = [np.abs(a).astype(np.float64) for a in xs], [np.abs(a).astype(np.float64) for a in gs]
    want = sum(x.astype(np.float64).T @ g for x, g in zip(xs, gs))        # (k, m)
    size = sum(x.T @ g for x, g in zip(*f))
    got = grads.get(pw).reshape(w.shape)
    assert np.all(np.abs((got.T if ta else got) - want) <= 2.0 ** -24 * (cols + 4) * (size + np.abs(want)))
    want = sum(g.astype(np.float64).sum(0) for g in gs) + 2.0 * b
    size = sum(g.sum(0) for g in f[1]) + 2 * np.abs(b)
    assert np.all(np.abs(grads.get(pb).reshape(m) - want) <= 2.0 ** -24 * (cols + 8) * (size + np.abs(want)))


@pytest.mark.parametrize("v,n,m,to,so", [(2048, 2, 4000, 0, 0), (2049, 3, 4007, 3, 3), (16385, 1, 8195, 1, 0),
                                         (65535, 1, 4001, 7, 7), (300, 33, 131073, 0, 0), (2048, 3, 4003, 4, 0), (2048, 3, 4009, 1, 3),
                                         (2048, 257, 5119, 0, 0), (2048, 257, 5120, 0, 0)])
def test_lookup_table_inverts_an_ascending_cdf(hip, v, n, m, to, so):
    """The inverse table of nchip_cdf_lookup, with columns that start `to` / `so` elements off a 16-byte
    boundary: runs of one target and of thousands, entries that share a value (the last one's
    symbol), a first entry above zero (symbol 0 below it)."""
    rng, lib = np.random.default_rng(v), C.CDLL(hip.lib._name)
    c = np.sort(rng.integers(0, 65536, (n, v)) if v > 1000 else 65535 * rng.random((n, v)) ** 8, axis=1).astype(np.uint16)
    t = rng.integers(0, 65536, (n, m)).astype(np.uint16)
    t[:, :3], t[:, -2:] = [[0, 65535, c[0, v // 2]]], [[c[0, 0], 65535]]
    c_t, t_t = hip.tensor(c), hip.tensor(np.concatenate([np.zeros(to, np.uint16), t.ravel()]))
    s_t = hip.tensor(np.full(so + n * m + 8, 0xabcd, np.uint16))
    ptr = [C.c_void_p(hip.nc_tensor_get_ptr(x, None) + o) for x, o in ((c_t, 0), (t_t, 2 * to), (s_t, 2 * so))]
    assert lib.nchip_cdf_lookup(C.c_void_p(hip.nc_context_stream(hip.ctx)), *ptr, C.c_int(v), C.c_int64(m), C.c_int64(n)) == 0
    got = hip.numpy(s_t)
    assert (got[:so] == 0xabcd).all() and (got[so + n * m:] == 0xabcd).all()
    want = [np.maximum(np.searchsorted(c[r], t[r], side="right") - 1, 0) for r in range(n)]
    assert np.array_equal(got[so:so + n * m].reshape(n, m), want)
    for x in (c_t, t_t, s_t):
        hip.free(x)


@pytest.mark.parametrize("cls,ta,tb,m,n,k,batch,ldc", [(10, 0, 0, 100, 67, 288, 40, 100), (10, 1, 0, 101, 68, 320, 40, 101), (10, 0, 1, 100, 68, 288, 40, 103),
                                                       (10, 1, 1, 99, 64, 288, 44, 100), (4, 0, 0, 132, 67, 32, 80, 132), (4, 1, 0, 133, 66, 96, 80, 133),
                                                       (4, 0, 1, 136, 72, 160, 70, 136), (7, 1, 0, 131, 129, 64, 130, 132), (7, 0, 1, 132, 132, 32, 130, 132),
                                                       (7, 0, 0, 260, 130, 128, 90, 260)])
def test_fp32_products_staged_by_dma_keep_the_sums_of_their_class(hip, cls, ta, tb, m, n, k, batch, ldc):
    """Partial tiles in both directions, fewer and more stages of 32 k than are in flight: the bits of the
    tile kernel of the same class, with bias, activation and the pre-activation kept."""
    lib, rng = C.CDLL(hip.lib._name), np.random.default_rng(m * k + n)
    p, i, j, f = C.c_void_p, C.c_int, C.c_int64, C.c_float
    lib.nchip_gemm2.argtypes = [p, i, i, i, i, i, f, p, j, j, j, p, j, j, j, f, p, j, j, j, i, i, p, i, p, i, i, p]
    a, b = rng.standard_normal((batch, m, k) if ta else (batch, k, m)), rng.standard_normal((batch, k, n) if tb else (batch, n, k))
    a_t, b_t, bias_t = (hip.tensor(x.astype(np.float32)) for x in (a, b, rng.standard_normal(m)))
    ptr = lambda t: p(hip.nc_tensor_get_ptr(t, None))
    got = []
    for forced in (0, cls):
        c_t, pre_t = (hip.tensor(np.full((batch, n, ldc), 7.0, np.float32)) for _ in range(2))
        lib.nchip_gemm_force_config(forced)
        rc = lib.nchip_gemm2(p(hip.nc_context_stream(hip.ctx)), ta, tb, m, n, k, 1.0, ptr(a_t), k if ta else m, m * k, 0, ptr(b_t),
                             n if tb else k, n * k, 0, 0.0, ptr(c_t), ldc, n * ldc, 0, batch, 1, ptr(bias_t), 1, ptr(pre_t), 0, 1, None)
        lib.nchip_gemm_force_config(0)
        assert rc == 0
        got.append([hip.numpy(c_t), hip.numpy(pre_t)])
        hip.free(c_t, pre_t)
    assert all(np.array_equal(x, y) for x, y in zip(*got))
    assert all((x[:, :, m:] == 7.0).all() for x in got[0])
    hip.free(a_t, b_t, bias_t)


@pytest.mark.parametrize("cls,ta,tb,m,n,k,batch,ksplit", [(10, 0, 0, 100, 68, 64, 60, 3), (10, 0, 1, 100, 68, 128, 60, 2), (10, 1, 0, 99, 67, 128, 60, 5),
                                                          (4, 0, 0, 132, 67, 64, 24, 3), (4, 1, 1, 132, 68, 96, 40, 2), (7, 0, 0, 260, 130, 64, 29, 3),
                                                          (7, 0, 1, 132, 132, 256, 9, 15), (7, 1, 0, 131, 129, 192, 64, 2)])
def test_fp32_products_split_over_k_under_dma(hip, cls, ta, tb, m, n, k, batch, ksplit):
    """Chunks of one stage and of several, and splits into more chunks than k has, whose last ones are empty
    and add nothing: the bits of the tile kernel of the same class, and float64 within a rounding per addition."""
    lib, rng = C.CDLL(hip.lib._name), np.random.default_rng(m * k + n)
    p, i, j, f = C.c_void_p, C.c_int, C.c_int64, C.c_float
    lib.nchip_gemm2.argtypes = [p, i, i, i, i, i, f, p, j, j, j, p, j, j, j, f, p, j, j, j, i, i, p, i, p, i, i, p]
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((batch, m, k) if ta else (batch, k, m), (batch, k, n) if tb else (batch, n, k)))
    a_t, b_t = hip.tensor(a), hip.tensor(b)
    ws_t = hip.tensor(np.full(batch * ksplit * m * n, 3.0, np.float32))
    ptr = lambda t: p(hip.nc_tensor_get_ptr(t, None))
    got = []
    for forced in (0, cls):
        c_t = hip.tensor(np.full((batch, n, m), 7.0, np.float32))
        lib.nchip_gemm_force_config(forced)
        rc = lib.nchip_gemm2(p(hip.nc_context_stream(hip.ctx)), ta, tb, m, n, k, 1.0, ptr(a_t), k if ta else m, m * k, 0, ptr(b_t),
                             n if tb else k, n * k, 0, 0.0, ptr(c_t), m, n * m, 0, batch, 1, None, 0, None, 0, ksplit, ptr(ws_t))
        lib.nchip_gemm_force_config(0)
        assert rc == 0
        got.append(hip.numpy(c_t, free=True))
    hip.free(a_t, b_t, ws_t)
    x = (a.transpose(0, 2, 1) if ta else a).astype(np.float64)  # (k, m)
    y = (b.transpose(0, 2, 1) if tb else b).astype(np.float64)  # (n, k)
    assert np.array_equal(*got)
    assert np.all(np.abs(got[0] - y @ x) <= 2.0 ** -24 * (k + 1) * (np.abs(y) @ np.abs(x)))


@pytest.mark.parametrize("m,n,k", [(132, 8200, 64), (100, 4100, 96)])
def test_fp32_activation_gradient_products_leave_their_row_sums_under_dma(hip, m, n, k):
    """nchip_gemm_dact_rowsum through the 128x64 and the two-group 64x64 tiles: the partial rows add up to
    the row sums of C (16 or 8 roundings a partial row, then the sum in float64)."""
    lib, rng = C.CDLL(hip.lib._name), np.random.default_rng(n)
    p, i, j = C.c_void_p, C.c_int, C.c_int64
    lib.nchip_gemm_dact_rowsum.argtypes = [p, i, i, i, i, i, C.c_float, p, j, p, j, p, j, p, i, i, i, p, p, C.POINTER(i)]
    w, dy, pre = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (n, k), (n, m)))
    rows, written = lib.nchip_gemm_rowsum_rows(n), C.c_int(0)
    w_t, dy_t, pre_t, c_t, rs_t = (hip.tensor(x) for x in (w, dy, pre, np.zeros((n, m), np.float32), np.full((rows, m), 9.0, np.float32)))
    ptr = lambda t: p(hip.nc_tensor_get_ptr(t, None))
    assert lib.nchip_gemm_dact_rowsum(p(hip.nc_context_stream(hip.ctx)), 1, 0, m, n, k, 1.0, ptr(w_t), k, ptr(dy_t), k, ptr(c_t), m,
                                      ptr(pre_t), 2, 0, 1, None, ptr(rs_t), C.byref(written)) == 0
    c, rs = hip.numpy(c_t).astype(np.float64), hip.numpy(rs_t).astype(np.float64)
    want = (dy.astype(np.float64) @ w.astype(np.float64).T) * (pre > 0)
    assert np.all(np.abs(c - want) <= 2.0 ** -24 * (k + 1) * (np.abs(dy) @ np.abs(w).T))
    assert 0 < written.value <= rows and np.all(np.abs(rs[: written.value].sum(0) - c.sum(0)) <= 2.0 ** -24 * 16 * np.abs(c).sum(0))
    hip.free(w_t, dy_t, pre_t, c_t, rs_t)


@pytest.mark.parametrize("cfg,precision", [(4, 0), (7, 0), (9, 0), (10, 0), (30, 0), (4, 1), (7, 1), (9, 1), (10, 1)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(131, 67, 257), (1, 130, 96), (129, 2, 193), (130, 3, 385), (128, 64, 97)])
def test_tile_products_at_any_alignment(hip, cfg, precision, ta, tb, m, n, k):
    """Partial tiles, columns that are no multiple of 4 floats apart and a base 4 bytes off a 16-byte unit: stages
    without guards up to the last one of a range, whose loads must not pass the operands' ends (they end
    with their buffers).  Operands are bf16 values, so both precisions form the same products; bound: a
    rounding per addition."""
    lib, rng = C.CDLL(hip.lib._name), np.random.default_rng(m * k + n)
    p, i, j, f = C.c_void_p, C.c_int, C.c_int64, C.c_float
    lib.nchip_gemm2.argtypes = [p, i, i, i, i, i, f, p, j, j, j, p, j, j, j, f, p, j, j, j, i, i, p, i, p, i, i, p]
    a, b = rng.standard_normal((m, k) if ta else (k, m)), rng.standard_normal((k, n) if tb else (n, k))
    a, b = ((x.astype(np.float32).view(np.uint32) & 0xffff0000).view(np.float32) for x in (a, b))
    a_t, b_t = (hip.tensor(np.concatenate([[np.nan], x.ravel()]).astype(np.float32)) for x in (a, b))
    c_t = hip.tensor(np.full((n, m), 7.0, np.float32))
    ptr = lambda t, skip=0: p(hip.nc_tensor_get_ptr(t, None) + 4 * skip)
    lib.nchip_gemm_force_config(cfg)
    rc = lib.nchip_gemm2(p(hip.nc_context_stream(hip.ctx)), ta, tb, m, n, k, 1.0, ptr(a_t, 1), k if ta else m, 0, 0, ptr(b_t, 1),
                         n if tb else k, 0, 0, 0.0, ptr(c_t), m, 0, 0, 1, 1, None, 0, None, precision, 1, None)
    lib.nchip_gemm_force_config(0)
    assert rc == 0
    x, y = (a.T if ta else a).astype(np.float64), (b.T if tb else b).astype(np.float64)  # (k, m), (n, k)
    assert np.all(np.abs(hip.numpy(c_t) - y @ x) <= 2.0 ** -24 * (k + 1) * (np.abs(y) @ np.abs(x)))
    hip.free(a_t, b_t, c_t)


@pytest.mark.parametrize("m,k,first,second", [(37, 21, 5, 3), (130, 70, 33, 31), (129, 131, 257, 65), (64, 128, 100, 320), (132, 36, 32, 1)])
@pytest.mark.parametrize("bf16", [0, 1])
def test_postponed_gradient_of_a_weight_used_over_two_widths(hip, pkg, m, k, first, second, bf16):
    """A weight used over two ranges of columns: one problem of the grouped launch where the range reached first
    (the later term's) is a multiple of 64, else two products.  Inputs are bf16 values; bound: a rounding per
    addition."""
    B, rng = pkg.binding, np.random.default_rng(m + first)
    bf = lambda *s: (rng.standard_normal(s).astype(np.float32).view(np.uint32) & 0xffff0000).view(np.float32)
    xs, gs = [bf(c, k) for c in (first, second)], [bf(c, m) for c in (first, second)]
    nc = B.NC(hip.lib._name, use_device=True)
    nc.nc_set_deferred_weight_grad(nc.ctx, 1)
    nc.nc_set_matmul_bf16(nc.ctx, bf16)
    h, _ = nc.param(np.zeros((k, m), np.float32))
    sp = B.SGDOptParams(algo=B.SGD_OPT_BASIC, lr=1.0)
    opt = nc.nc_sgd_opt_init(nc.ctx, C.byref(sp))
    nc.nc_sgd_opt_set_all(C.byref(nc.plist), opt)
    loss = None
    for x, g in zip(xs, gs):
        term = nc.nc_sum(nc.nc_mul(nc.nc_matmul(nc.dup(h.value), nc.tensor(x)), nc.tensor(g)))
        loss = term if loss is None else nc.nc_add(loss, term)
    nc.lib.nc_backward(loss, nc.nc_new_f32(nc.dev, 1.0), C.cast(nc.lib.sgd_opt_update_var, B.PARAM_UPDATE_FUNC), 0)
    nc.free(loss)
    nc.nc_sgd_opt_update(opt)
    got = -nc.numpy(h.value)
    nc.nc_sgd_opt_set_all(C.byref(nc.plist), None)
    nc.nc_sgd_opt_end(opt)
    nc.close()
    want = sum(x.astype(np.float64).T @ g for x, g in zip(xs, gs))
    size = sum(np.abs(x).astype(np.float64).T @ np.abs(g) for x, g in zip(xs, gs))
    assert np.all(np.abs(got - want) <= 2.0 ** -24 * (first + second + 2) * size)


@pytest.mark.parametrize("m,k,later,earlier", [(37, 21, 5, 3), (130, 70, 33, 31), (352, 352, 585, 481), (128, 128, 64, 100), (128, 256, 448, 33), (128, 128, 33, 64), (64, 96, 33, 1100)])
@pytest.mark.parametrize("bf16", [0, 1])
def test_postponed_gradient_over_two_widths_is_the_sum_of_two_products(hip, pkg, m, k, later, earlier, bf16):
    """A weight whose use that is reached first (the later term of the loss) has a number of columns that is no
    multiple of 64: the bits of the postponed gradient of that use alone plus the product of the other
    one alone, each in the class of its own shape."""
    B, rng = pkg.binding, np.random.default_rng(m + later)
    xs, gs = ([rng.standard_normal((c, d)).astype(np.float32) for c in (earlier, later)] for d in (k, m))

    def gradient(uses, postponed):
        nc = B.NC(hip.lib._name, use_device=True)
        nc.nc_set_deferred_weight_grad(nc.ctx, postponed)
        nc.nc_set_matmul_bf16(nc.ctx, bf16)
        h, _ = nc.param(np.zeros((k, m), np.float32))
        sp = B.SGDOptParams(algo=B.SGD_OPT_BASIC, lr=1.0)
        opt = nc.nc_sgd_opt_init(nc.ctx, C.byref(sp))
        nc.nc_sgd_opt_set_all(C.byref(nc.plist), opt)
        loss = None
        for u in uses:
            term = nc.nc_sum(nc.nc_mul(nc.nc_matmul(nc.dup(h.value), nc.tensor(xs[u])), nc.tensor(gs[u])))
            loss = term if loss is None else nc.nc_add(loss, term)
        nc.lib.nc_backward(loss, nc.nc_new_f32(nc.dev, 1.0), C.cast(nc.lib.sgd_opt_update_var, B.PARAM_UPDATE_FUNC), 0)
        nc.free(loss)
        nc.nc_sgd_opt_update(opt)
        got = -nc.numpy(h.value)
        nc.nc_sgd_opt_set_all(C.byref(nc.plist), None)
        nc.nc_sgd_opt_end(opt)
        nc.close()
        return got

    # (the later term's use is reached first; with 64 or 448 columns it is joined by the other as a second range)
    both, alone, other = gradient((0, 1), 1), gradient((1,), 1), gradient((0,), 0)
    if later % 64:
        assert np.array_equal(both, alone + other)
    else:
        want, size = (sum(f(x).T @ f(g) for x, g in zip(xs, gs)) for f in (lambda a: a.astype(np.float64), lambda a: np.abs(a).astype(np.float64)))
        assert np.all(np.abs(both - want) <= (2.0 ** -7 * bf16 + 2.0 ** -24 * (later + earlier + 2)) * size)
