"""The AMR transfer operators on the device against the oracle, through the
C-ABI: the reference's single-call forms (faceUnknowns*/volumeUnknowns*
Prolongation/Restriction) at orders 1..5 over one and two levels, and the
batched device forms over whole coarse/fine block sets, restriction
accumulating several children in list order.  Bar: 1e-12 of each array's
scale (the device sums the tensor-product operator direction by direction,
the reference node by node: the same linear map, other rounding).
"""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.abs(np.asarray(a) - np.asarray(b)).max() / max(np.abs(np.asarray(b)).max(), 1e-300)


def _solvers(exa, oracle, order, nvar=5, npar=1):
    return exa.euler_solver(order, npar=npar), oracle.make_solver(order, nvar=nvar, npar=npar)


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("level_delta", [1, 2])
def test_single_volume_transfers_vs_oracle(exa, oracle, order, level_delta):
    print(f"case: volume prolongation/restriction N={order} levels={level_delta}", flush=True)
    rng = np.random.default_rng(order * 7 + level_delta)
    s, os_ = _solvers(exa, oracle, order)
    B, D = order + 1, 6
    n = 3 ** level_delta
    for sub in [(0, 0, 0), (n - 1, 0, 1), tuple(rng.integers(0, n, 3))]:
        uc = rng.standard_normal(B ** 3 * D)
        dev = exa.volume_unknowns_prolongation(s, uc, 1, 1 + level_delta, sub)
        ref = oracle.volume_unknowns_prolongation(os_, uc, 1, 1 + level_delta, sub)
        assert _rel(dev, ref) <= 1e-12, sub
        uf, acc = rng.standard_normal(B ** 3 * D), rng.standard_normal(B ** 3 * D)
        dev = exa.volume_unknowns_restriction(s, acc, uf, 1, 1 + level_delta, sub)
        ref = oracle.volume_unknowns_restriction(os_, acc, uf, 1, 1 + level_delta, sub)
        assert _rel(dev, ref) <= 1e-12, sub


@pytest.mark.parametrize("order", [1, 3, 5])
@pytest.mark.parametrize("level_delta", [1, 2])
def test_single_face_transfers_vs_oracle(exa, oracle, order, level_delta):
    print(f"case: face prolongation/restriction N={order} levels={level_delta}", flush=True)
    rng = np.random.default_rng(100 + order * 7 + level_delta)
    s, os_ = _solvers(exa, oracle, order)
    B, D, V = order + 1, 6, 5
    n = 3 ** level_delta
    for sub in [(0, 0), (n - 1, 1), tuple(rng.integers(0, n, 2))]:
        qc, fc = rng.standard_normal(B * B * D), rng.standard_normal(B * B * V)
        dq, df = exa.face_unknowns_prolongation(s, qc, fc, 0, level_delta, sub)
        rq, rf = oracle.face_unknowns_prolongation(os_, qc, fc, 0, level_delta, sub)
        assert _rel(dq, rq) <= 1e-12 and _rel(df, rf) <= 1e-12, sub
        qf, ff = rng.standard_normal(B * B * D), rng.standard_normal(B * B * V)
        dq, df = exa.face_unknowns_restriction(s, qc, fc, qf, ff, 0, level_delta, sub)
        rq, rf = oracle.face_unknowns_restriction(os_, qc, fc, qf, ff, 0, level_delta, sub)
        assert _rel(dq, rq) <= 1e-12 and _rel(df, rf) <= 1e-12, sub


def test_single_call_level_rules(exa):
    s = exa.euler_solver(3, npar=1)
    uc = np.ones(64 * 6)
    uf = np.full(64 * 6, 7.0)
    # prolongation over zero levels leaves the fine block as it was (the reference's loop does not run)
    assert np.array_equal(exa.volume_unknowns_prolongation(s, uc, 2, 2, (0, 0, 0), uF=uf), uf)
    with pytest.raises(exa.ExaError):  # restriction needs a finer level
        exa.volume_unknowns_restriction(s, uc, uf, 2, 2, (0, 0, 0))
    with pytest.raises(exa.ExaError):  # subinterval index beyond 3^levels
        exa.volume_unknowns_prolongation(s, uc, 0, 1, (3, 0, 0))


def _children(nc, level_delta):
    """Fine blocks of an nc^3 coarse grid refined by 3^level_delta: items
    (fine, coarse, sx, sy, sz) in coarse-major order, and the CSR pointer."""
    r = 3 ** level_delta
    nf = nc * r
    items, ptr = [], [0]
    for c in range(nc ** 3):
        ci, cj, ck = c % nc, (c // nc) % nc, c // (nc * nc)
        for sz, sy, sx in itertools.product(range(r), repeat=3):
            fi, fj, fk = ci * r + sx, cj * r + sy, ck * r + sz
            items.append((fi + nf * (fj + nf * fk), c, sx, sy, sz))
        ptr.append(len(items))
    return np.array(items, dtype=np.int32), np.array(ptr, dtype=np.int32)


@pytest.mark.parametrize("order,level_delta", [(3, 1), (2, 2), (5, 1)])
def test_volume_batches_vs_oracle(exa, oracle, order, level_delta):
    print(f"case: volume batches N={order} levels={level_delta}", flush=True)
    rng = np.random.default_rng(order + 10 * level_delta)
    s, os_ = _solvers(exa, oracle, order)
    B, D = order + 1, 6
    nc = 2
    items, ptr = _children(nc, level_delta)
    nfine = len(items)
    coarse = rng.standard_normal((nc ** 3, B ** 3 * D))
    d_coarse, d_fine = exa.DeviceArray(coarse), exa.DeviceArray(np.zeros((nfine, B ** 3 * D)))
    # prolongation items: (fine destination, coarse source, sub); restriction: (coarse, fine, sub)
    d_items, d_ptr = exa.DeviceArray(items), exa.DeviceArray(ptr)
    d_ritems = exa.DeviceArray(items[:, [1, 0, 2, 3, 4]])
    ms = exa.volume_prolongation_batch(s, d_fine, d_coarse, d_items, level_delta)
    assert ms > 0.0
    fine = d_fine.get()
    for it in items[:: max(1, nfine // 40)]:
        ref = oracle.volume_unknowns_prolongation(os_, coarse[it[1]], 0, level_delta, it[2:])
        assert _rel(fine[it[0]], ref) <= 1e-12
    # restriction: every coarse block gets its children added in list order
    fine_in = rng.standard_normal((nfine, B ** 3 * D))
    start = rng.standard_normal((nc ** 3, B ** 3 * D))
    d_fine_in, d_acc = exa.DeviceArray(fine_in), exa.DeviceArray(start)
    exa.volume_restriction_batch(s, d_acc, d_fine_in, d_ptr, d_ritems, level_delta)
    acc = d_acc.get()
    for c in range(nc ** 3):
        ref = start[c].copy()
        for it in items[ptr[c]:ptr[c + 1]]:
            ref = oracle.volume_unknowns_restriction(os_, ref, fine_in[it[0]], 0, level_delta, it[2:])
        assert _rel(acc[c], ref) <= 1e-12, c


def test_face_batches_vs_oracle(exa, oracle):
    print("case: face batches N=4 one level", flush=True)
    rng = np.random.default_rng(44)
    s, os_ = _solvers(exa, oracle, 4)
    B, D, V = 5, 6, 5
    ncf = 4  # coarse face blocks, each split into 9 fine face blocks
    items = np.array([(9 * c + 3 * b + a, c, a, b, 0) for c in range(ncf) for b in range(3) for a in range(3)],
                     dtype=np.int32)
    ptr = np.arange(0, 9 * ncf + 1, 9, dtype=np.int32)
    qc, fc = rng.standard_normal((ncf, B * B * D)), rng.standard_normal((ncf, B * B * V))
    d_qc, d_fc = exa.DeviceArray(qc), exa.DeviceArray(fc)
    d_qf, d_ff = exa.DeviceArray(np.zeros((9 * ncf, B * B * D))), exa.DeviceArray(np.zeros((9 * ncf, B * B * V)))
    d_items, d_ptr = exa.DeviceArray(items), exa.DeviceArray(ptr)
    d_ritems = exa.DeviceArray(items[:, [1, 0, 2, 3, 4]])
    exa.face_prolongation_batch(s, d_qf, d_ff, d_qc, d_fc, d_items, 1)
    qf, ff = d_qf.get(), d_ff.get()
    for it in items:
        rq, rf = oracle.face_unknowns_prolongation(os_, qc[it[1]], fc[it[1]], 0, 1, it[2:4])
        assert _rel(qf[it[0]], rq) <= 1e-12 and _rel(ff[it[0]], rf) <= 1e-12
    exa.face_restriction_batch(s, d_qc, d_fc, d_qf, d_ff, d_ptr, d_ritems, 1)
    q2, f2 = d_qc.get(), d_fc.get()
    for c in range(ncf):
        rq, rf = qc[c].copy(), fc[c].copy()
        for it in items[ptr[c]:ptr[c + 1]]:
            rq, rf = oracle.face_unknowns_restriction(os_, rq, rf, qf[it[0]], ff[it[0]], 0, 1, it[2:4])
        assert _rel(q2[c], rq) <= 1e-12 and _rel(f2[c], rf) <= 1e-12
    # prolongation then complete restriction onto zero blocks returns the coarse data
    z_q, z_f = exa.DeviceArray(np.zeros_like(qc)), exa.DeviceArray(np.zeros_like(fc))
    exa.face_restriction_batch(s, z_q, z_f, d_qf, d_ff, d_ptr, d_ritems, 1)
    assert _rel(z_q.get(), qc) <= 1e-11 and _rel(z_f.get(), fc) <= 1e-11


def test_batch_rejects_out_of_range_items(exa):
    s = exa.euler_solver(2, npar=1)
    blk = 27 * 6
    d_c, d_f = exa.DeviceArray(np.ones((2, blk))), exa.DeviceArray(np.zeros((3, blk)))
    bad = exa.DeviceArray(np.array([(0, 0, 0, 0, 0), (5, 0, 0, 0, 0), (1, 1, 3, 0, 0)], dtype=np.int32))
    with pytest.raises(exa.ExaError):
        exa.volume_prolongation_batch(s, d_f, d_c, bad, 1)
    assert np.allclose(d_f.get()[0], 1.0)  # the valid item ran
    bad_ptr = exa.DeviceArray(np.array([0, 7], dtype=np.int32))  # a range beyond the item list
    good = exa.DeviceArray(np.array([(0, 0, 0, 0, 0)], dtype=np.int32))
    with pytest.raises(exa.ExaError):
        exa.volume_restriction_batch(s, d_c, d_f, bad_ptr, good, 1)


def test_batch_rejects_repeated_destinations(exa, oracle):
    """A destination block named twice in one call (two prolongation items, or
    two restriction ranges) is written by one transfer only and the call fails."""
    print("case: repeated AMR destinations", flush=True)
    s, os_ = _solvers(exa, oracle, 2)
    blk = 27 * 6
    rng = np.random.default_rng(5)
    coarse = rng.standard_normal((2, blk))
    d_c, d_f = exa.DeviceArray(coarse), exa.DeviceArray(np.zeros((3, blk)))
    dup = exa.DeviceArray(np.array([(1, 0, 0, 0, 0), (2, 1, 1, 1, 1), (1, 1, 2, 0, 1)], dtype=np.int32))
    with pytest.raises(exa.ExaError):
        exa.volume_prolongation_batch(s, d_f, d_c, dup, 1)
    fine = d_f.get()
    assert np.array_equal(fine[0], np.zeros(blk))  # named by no item
    ref2 = oracle.volume_unknowns_prolongation(os_, coarse[1], 0, 1, (1, 1, 1))
    assert _rel(fine[2], ref2) <= 1e-12  # the unique destination is written
    cands = [oracle.volume_unknowns_prolongation(os_, coarse[0], 0, 1, (0, 0, 0)),
             oracle.volume_unknowns_prolongation(os_, coarse[1], 0, 1, (2, 0, 1))]
    assert min(_rel(fine[1], c) for c in cands) <= 1e-12  # exactly one of the two transfers landed
    # restriction: two ranges with the same destination
    start = rng.standard_normal((2, blk))
    d_acc = exa.DeviceArray(start)
    ritems = exa.DeviceArray(np.array([(0, 0, 0, 0, 0), (0, 1, 1, 0, 0), (1, 2, 2, 2, 2)], dtype=np.int32))
    rptr = exa.DeviceArray(np.array([0, 1, 2, 3], dtype=np.int32))
    d_fin = exa.DeviceArray(rng.standard_normal((3, blk)))
    with pytest.raises(exa.ExaError):
        exa.volume_restriction_batch(s, d_acc, d_fin, rptr, ritems, 1)
    # the same ranges with distinct destinations are accepted
    ok_items = exa.DeviceArray(np.array([(0, 0, 0, 0, 0), (0, 1, 1, 0, 0), (1, 2, 2, 2, 2)], dtype=np.int32))
    ok_ptr = exa.DeviceArray(np.array([0, 2, 3], dtype=np.int32))
    exa.volume_restriction_batch(s, exa.DeviceArray(start), d_fin, ok_ptr, ok_items, 1)


@pytest.mark.parametrize("order,nv,children", [(1, 5, (1, 3, 0, 27)), (2, 5, (4, 5, 1, 0)), (3, 5, (27, 2, 8, 9)),
                                               (4, 12, (5, 0, 4, 3)), (5, 5, (27, 1, 6, 0)), (5, 12, (3, 5, 0, 1))])
def test_batches_uneven_ranges_vs_oracle(exa, oracle, order, nv, children):
    """Both directions with 5 values per node and another count, destinations
    with no, few and many transfers (a destination's transfers run four at a
    time), a number of transfers that fills no whole workgroup."""
    print(f"case: AMR batches N={order} nv={nv} children={children}", flush=True)
    rng = np.random.default_rng(order * 100 + nv)
    s, os_ = (_solvers(exa, oracle, order, npar=0) if nv == 5 else
              (exa.elastic_solver(order), oracle.elastic_solver(order)))
    blk = (order + 1) ** 3 * nv
    nfine = sum(children)
    sub = rng.integers(0, 3, (nfine, 3))
    owner = np.repeat(np.arange(len(children)), children)
    order_ = rng.permutation(nfine)  # fine blocks in any order
    items = np.column_stack([order_, owner, sub]).astype(np.int32)
    ptr = np.concatenate([[0], np.cumsum(children)]).astype(np.int32)
    coarse = rng.standard_normal((len(children), blk))
    d_fine = exa.DeviceArray(np.zeros((nfine, blk)))
    exa.volume_prolongation_batch(s, d_fine, exa.DeviceArray(coarse), exa.DeviceArray(items), 1)
    fine = d_fine.get()
    for it in items:
        assert _rel(fine[it[0]], oracle.volume_unknowns_prolongation(os_, coarse[it[1]], 0, 1, it[2:])) <= 1e-12
    acc, d_acc = coarse.copy(), exa.DeviceArray(coarse)
    fine_in = rng.standard_normal((nfine, blk))
    exa.volume_restriction_batch(s, d_acc, exa.DeviceArray(fine_in), exa.DeviceArray(ptr),
                                 exa.DeviceArray(np.ascontiguousarray(items[:, [1, 0, 2, 3, 4]])), 1)
    for it in items:
        acc[it[1]] = oracle.volume_unknowns_restriction(os_, acc[it[1]], fine_in[it[0]], 0, 1, it[2:])
    assert _rel(d_acc.get(), acc) <= 1e-12


def _any_solver(exa, oracle, order, nv):
    return (exa.Solver(exa.PDE_EULER, order, nv, 0, exa.TERM_FLUX, 0, 0.9, exa.PRECISION_FP64, 0),
            oracle.make_solver(order, nvar=nv, npar=0))


# (order, values per node, transfers, levels): both sides of the lines between a
# thread per value, a workgroup and a wavefront per transfer
PROLONGATIONS = [(1, 1, 7, 3), (3, 4, 2100, 1), (2, 10, 2048, 1), (2, 10, 2049, 2), (3, 8, 1153, 1), (4, 8, 1152, 1),
                 (4, 8, 1153, 1), (3, 17, 500, 2), (5, 5, 512, 1), (5, 5, 513, 1), (5, 9, 513, 1), (5, 12, 600, 1),
                 (5, 12, 3, 2)]


@pytest.mark.parametrize("order,nv,count,levels", PROLONGATIONS)
def test_prolongation_forms(exa, oracle, order, nv, count, levels):
    """One long list against the same transfers in lists of 50, which take other
    forms of the kernel with the same sums in the same order (1e-14), and single
    transfers against the oracle."""
    print(f"case: AMR prolongation forms N={order} nv={nv} {count} transfers {levels} levels", flush=True)
    rng = np.random.default_rng(order * 1000 + nv + count)
    s, os_ = _any_solver(exa, oracle, order, nv)
    blk, r = (order + 1) ** 3 * nv, 3 ** levels
    coarse = rng.standard_normal((5, blk))
    items = np.column_stack([rng.permutation(count), rng.integers(0, 5, count),
                             rng.integers(0, r, (count, 3))]).astype(np.int32)
    d_c, d_f = exa.DeviceArray(coarse), exa.DeviceArray(np.zeros((count, blk)))
    exa.volume_prolongation_batch(s, d_f, d_c, exa.DeviceArray(items), levels)
    fine = d_f.get()
    d_g = exa.DeviceArray(np.zeros((count, blk)))
    for k in range(0, count, 50):
        exa.volume_prolongation_batch(s, d_g, d_c, exa.DeviceArray(items[k:k + 50]), levels)
    assert _rel(fine, d_g.get()) <= 1e-14
    for it in items[:: max(1, count // 5)]:
        ref = oracle.volume_unknowns_prolongation(os_, coarse[it[1]], 0, levels, it[2:])
        assert _rel(fine[it[0]], ref) <= 1e-12


@pytest.mark.parametrize("order,nv,count", [(2, 3, 40), (4, 8, 40), (4, 12, 40), (4, 8, 1300)])
def test_prolongation_forms_report_bad_items(exa, oracle, order, nv, count):
    """Every form skips an item out of range and writes a block named twice once,
    and the call fails."""
    print(f"case: AMR prolongation bad items N={order} nv={nv} {count} transfers", flush=True)
    rng = np.random.default_rng(count + nv)
    s, os_ = _any_solver(exa, oracle, order, nv)
    blk = (order + 1) ** 3 * nv
    coarse = rng.standard_normal((2, blk))
    items = np.column_stack([np.arange(count), rng.integers(0, 2, count), rng.integers(0, 3, (count, 3))])
    items = items.astype(np.int32)
    items[7, 0] = count  # no such block
    items[9, 3] = 3      # no such subcell
    items[20, 0] = 19    # block 19 twice
    d_c, d_f = exa.DeviceArray(coarse), exa.DeviceArray(np.zeros((count, blk)))
    with pytest.raises(exa.ExaError):
        exa.volume_prolongation_batch(s, d_f, d_c, exa.DeviceArray(items), 1)
    fine = d_f.get()
    assert not fine[[7, 9, 20]].any()
    ref = [oracle.volume_unknowns_prolongation(os_, coarse[it[1]], 0, 1, it[2:]) for it in items[[18, 19, 20]]]
    assert _rel(fine[18], ref[0]) <= 1e-12
    assert min(_rel(fine[19], ref[1]), _rel(fine[19], ref[2])) <= 1e-12


@pytest.mark.parametrize("order,nv,children,levels", [(4, 13, (9, 0, 4, 1), 1), (5, 8, (1, 5, 0, 27), 1),
                                                      (5, 12, (3, 0, 6, 1), 2), (3, 25, (2, 5, 1, 3), 1)])
def test_restriction_of_large_blocks_vs_oracle(exa, oracle, order, nv, children, levels):
    """Blocks of which 64 KiB hold four and a destination, and of which they do
    not (a workgroup per transfer); an item out of range is skipped."""
    print(f"case: AMR restriction N={order} nv={nv} children={children} levels={levels}", flush=True)
    rng = np.random.default_rng(order + nv)
    s, os_ = _any_solver(exa, oracle, order, nv)
    blk, n = (order + 1) ** 3 * nv, sum(children)
    items = np.column_stack([np.repeat(np.arange(len(children)), children), rng.permutation(n),
                             rng.integers(0, 3 ** levels, (n, 3))]).astype(np.int32)
    ptr = np.concatenate([[0], np.cumsum(children)]).astype(np.int32)
    coarse, fine = rng.standard_normal((len(children), blk)), rng.standard_normal((n, blk))
    for bad in (None, 1):
        it_run = items.copy()
        if bad is not None:
            it_run[bad, 1] = n  # no such block
        d_acc = exa.DeviceArray(coarse)
        call = (s, d_acc, exa.DeviceArray(fine), exa.DeviceArray(ptr), exa.DeviceArray(it_run), levels)
        if bad is None:
            exa.volume_restriction_batch(*call)
        else:
            with pytest.raises(exa.ExaError):
                exa.volume_restriction_batch(*call)
        acc = coarse.copy()
        for k, it in enumerate(items):
            if k != bad:
                acc[it[0]] = oracle.volume_unknowns_restriction(os_, acc[it[0]], fine[it[1]], 0, levels, it[2:])
        assert _rel(d_acc.get(), acc) <= 1e-12
