"""GPU all-pairs gravity (libncg.so) against the oracle.

NCG_F64_EXACT must be bit-identical to the reference's vector_field; the FP64-
fast form must agree to FP64 rounding; the mixed form must stay within the
north-star tolerance of 1e-6 max relative error on the mutual acceleration.
"""
import os

import numpy as np
import pytest

import oracle_lib as orc
from ncorpion_amd import ic

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def rel_err(a, ref):
    """Per-body |a - ref| / |ref| (max over bodies) and normwise max |da| / rms|ref|."""
    d = np.linalg.norm(a - ref, axis=1)
    r = np.linalg.norm(ref, axis=1)
    return float(np.max(d / r)), float(np.max(d) / np.sqrt(np.mean(r * r)))


@pytest.mark.parametrize("name", ["vf_bf_g1_n3", "vf_bf_g1_n257_holes", "vf_bf_soft_n64",
                                  "vf_bf_nocm_n200", "vf_c3_n4096"])
def test_exact_matches_reference_golden(ctx, name):
    g = dict(np.load(os.path.join(GOLD, name + ".npz")))
    c8 = g.get("central")
    cen = (c8[0], c8[1], c8[2], c8[6]) if c8 is not None else None
    ex = g.get("exists")
    acc, cm = ctx.gravity_allpairs(g["bodies"], ex, cen, float(g["G"]), float(g["soft"]), "exact")
    keep = ex.astype(bool) if ex is not None else np.ones(len(acc), bool)
    assert np.array_equal(bits(acc[keep]), bits(g["acc"][keep]))
    if cen is not None:
        assert np.array_equal(bits(cm), bits(g["cm_acc"]))


@pytest.mark.parametrize("n,seed,soft,central,holes", [
    (1, 0, 0.0, True, False), (2, 1, 0.0, False, False), (255, 2, 0.0, True, True),
    (256, 3, 0.3, True, False), (257, 4, 1e-6, False, True), (1000, 5, 0.0, True, True),
    (3001, 6, 0.05, True, False)])
def test_exact_bitwise_random(ctx, n, seed, soft, central, holes):
    b = ic.disk(n, seed=seed, mass=1e-6, radius=1e-3)
    b[:, 6] *= np.random.default_rng(seed).uniform(0.5, 2.0, n)
    ex = None
    if holes:
        ex = (np.random.default_rng(seed + 9).uniform(size=n) > 0.15).astype(np.int32)
    cen = (1e-3, 2e-3, -1e-3, 1.0) if central else None
    ref, rcm = orc.vector_field_brute(b, ex, cen, 1.0, soft)
    acc, cm = ctx.gravity_allpairs(b, ex, cen, 1.0, soft, "exact")
    keep = ex.astype(bool) if ex is not None else np.ones(n, bool)
    assert np.array_equal(bits(acc[keep]), bits(ref[keep]))
    if central:
        assert np.array_equal(bits(cm), bits(rcm))


def test_holes_left_untouched(ctx):
    b = ic.disk(100, seed=7)
    ex = np.ones(100, np.int32)
    ex[::7] = 0
    acc = np.full((100, 3), 123.0)
    ctx.gravity_allpairs(b, ex, (0, 0, 0, 1.0), 1.0, 0.0, "exact", acc=acc)
    assert np.all(acc[~ex.astype(bool)] == 123.0)


def c3_disk(n, seed=0):
    m, R = ic.disk_c3_masses(n, seed)
    return ic.disk(n, seed=seed, masses=m, radii=R)


# 1000 and 4096 run the direct form (up to 4096 bodies), 4097 and 8192 the
# tiled one.
@pytest.mark.parametrize("n", [1000, 4096, 4097, 8192])
def test_fast64_matches_oracle(ctx, n):
    b = c3_disk(n, 11)
    ref, rcm = orc.vector_field_brute(b, None, None, 1.0, 1e-6)
    acc, _ = ctx.gravity_allpairs(b, None, None, 1.0, 1e-6, "fast64")
    mx, nw = rel_err(acc, ref)
    assert mx < 1e-12, mx
    # With the central body the reference adds n mutual terms one by one onto
    # an O(1) central term, so its own rounding is ~sqrt(n) * 1e-16 of |a|.
    ref2, rcm2 = orc.vector_field_brute(b, None, (0, 0, 0, 1.0), 1.0, 1e-6)
    acc2, cm2 = ctx.gravity_allpairs(b, None, (0, 0, 0, 1.0), 1.0, 1e-6, "fast64")
    assert np.max(np.abs(acc2 - ref2) / np.abs(ref2).max()) < 4e-16 * np.sqrt(n) + 1e-15
    assert np.allclose(cm2, rcm2, rtol=1e-12, atol=0)


@pytest.mark.parametrize("n", [1000, 4096, 4097, 16384])
def test_mixed_within_tolerance(ctx, n):
    # Mutual part only (the central term is FP64 in every form).
    b = c3_disk(n, 12)
    ref, _ = orc.vector_field_brute(b, None, None, 1.0, 1e-6)
    acc, _ = ctx.gravity_allpairs(b, None, None, 1.0, 1e-6, "mixed")
    mx, nw = rel_err(acc, ref)
    assert mx <= 1e-6, (mx, nw)


def test_mixed_with_holes_and_softening(ctx):
    b = ic.disk(3000, seed=13, mass=1e-7, radius=5e-3)
    ex = (np.random.default_rng(1).uniform(size=3000) > 0.2).astype(np.int32)
    ref, rcm = orc.vector_field_brute(b, ex, (0, 0, 0, 1.0), 1.0, 0.5)
    acc, cm = ctx.gravity_allpairs(b, ex, (0, 0, 0, 1.0), 1.0, 0.5, "mixed")
    keep = ex.astype(bool)
    refm, _ = orc.vector_field_brute(b, ex, None, 1.0, 0.5)
    accm, _ = ctx.gravity_allpairs(b, ex, None, 1.0, 0.5, "mixed")
    mx, _ = rel_err(accm[keep], refm[keep])
    assert mx <= 1e-6, mx
    assert np.allclose(cm, rcm, rtol=1e-12, atol=0)


def test_device_entry_point_matches_host(ctx):
    import torch
    b = c3_disk(5000, 14)
    acc_h, cm_h = ctx.gravity_allpairs(b, None, (0, 0, 0, 1.0), 1.0, 1e-6, "mixed")
    bt = torch.from_numpy(b).cuda()
    at = torch.zeros((5000, 3), dtype=torch.float64, device="cuda")
    ct = torch.zeros(3, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ctx.gravity_allpairs_dev(bt, at, None, (0, 0, 0, 1.0), 1.0, 1e-6, "mixed", ct)
    ctx.synchronize()
    assert np.array_equal(at.cpu().numpy(), acc_h)
    assert np.array_equal(ct.cpu().numpy(), cm_h)


@pytest.mark.parametrize("n", [1000, 4096, 4097, 8192])
@pytest.mark.parametrize("prec,tol", [("fast64", 1e-12), ("mixed", 1e-6)])
def test_no_softening_with_large_gm(ctx, n, prec, tol):
    # Without softening (NcorpiON's default) a body's pair with itself has
    # r = 0.  With G m far above 1 (SI or cgs units: here G m spans 1e7..1e9)
    # that term must still add exactly nothing rather than inf * 0.  Both
    # sides of the direct form's 4096-body limit.
    b = c3_disk(n, 15)
    G = 1e18
    ref, _ = orc.vector_field_brute(b, None, None, G, 0.0)
    acc, _ = ctx.gravity_allpairs(b, None, None, G, 0.0, prec)
    assert np.all(np.isfinite(acc))
    mx, _ = rel_err(acc, ref)
    assert mx <= tol, mx


def test_exact_device_entry_point_cm_acc_in_reference_order(ctx):
    # The device entry point sums CM_acc body by body as vector_field does
    # (physics.c:141-146): bit-identical to the oracle, holes included.
    import torch
    n = 3000
    b = ic.disk(n, seed=16, mass=1e-6, radius=1e-3)
    b[:, 6] *= np.random.default_rng(16).uniform(0.5, 2.0, n)
    ex = (np.random.default_rng(17).uniform(size=n) > 0.1).astype(np.int32)
    cen = (1e-3, 2e-3, -1e-3, 1.0)
    ref, rcm = orc.vector_field_brute(b, ex, cen, 1.0, 0.01)
    bt = torch.from_numpy(b).cuda()
    et = torch.from_numpy(ex).cuda()
    at = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
    ct = torch.zeros(3, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ctx.gravity_allpairs_dev(bt, at, et, cen, 1.0, 0.01, "exact", ct)
    ctx.synchronize()
    keep = ex.astype(bool)
    assert np.array_equal(bits(at.cpu().numpy()[keep]), bits(ref[keep]))
    assert np.array_equal(bits(ct.cpu().numpy()), bits(rcm))


def test_empty_and_single(ctx):
    acc, cm = ctx.gravity_allpairs(np.zeros((0, 8)), None, (0, 0, 0, 1.0), 1.0, 0.0, "mixed")
    assert acc.shape == (0, 3)
    b = np.array([[1.0, 0, 0, 0, 0, 0, 1e-3, 1e-3]])
    for p in ("exact", "fast64", "mixed"):
        acc, _ = ctx.gravity_allpairs(b, None, (0, 0, 0, 2.0), 1.0, 0.0, p)
        assert acc[0, 0] == -2.0 and acc[0, 1] == 0.0


def central_start(b, ex, cen, G):
    """The central term of vector_field (physics.c:121-136) in numpy, which
    rounds each operation as the reference does: ((-mu) DX) / r^3."""
    cx, cy, cz, M = cen
    mu = G * M
    DX, DY, DZ = b[:, 0] - cx, b[:, 1] - cy, b[:, 2] - cz
    rk = np.sqrt(DX * DX + DY * DY + DZ * DZ)
    r3 = rk * rk * rk
    st = np.stack([-mu * DX / r3, -mu * DY / r3, -mu * DZ / r3], axis=1)
    st[~ex] = 0.0
    return st


@pytest.mark.parametrize("n,prec", [(1000, "exact"), (40000, "exact"), (1000, "fast64"),
                                    (8192, "fast64"), (8192, "mixed")])
def test_start_values_equal_central_term(ctx, n, prec):
    """ncg_gravity_allpairs_from with the central term as the start values
    equals ncg_gravity_allpairs with the central body: bit for bit in the
    exact form (both paths of the exact kernel, n below and above 32,768),
    within the form's tolerance in the others (which add the start values
    after their sums)."""
    rng = np.random.default_rng(n)
    b = ic.disk(n, seed=n, mass=1e-8, radius=2e-4)
    ex = np.ones(n, np.int32)
    ex[rng.choice(n, n // 50, replace=False)] = 0
    cen = (1e-3, -2e-3, 0.0, 1.0)
    G, soft = 1.0, 0.25
    ref, _ = ctx.gravity_allpairs(b, ex, cen, G, soft, prec)
    got = ctx.gravity_allpairs_from(b, central_start(b, ex != 0, cen, G), ex, G, soft, prec)
    live = ex != 0
    if prec == "exact":
        assert np.array_equal(bits(got[live]), bits(ref[live]))
    else:
        tol = 1e-12 if prec == "fast64" else 1e-6
        assert rel_err(got[live], ref[live])[0] < tol


def _exact_edge_bodies(n, kind):
    rng = np.random.default_rng(n + len(kind))
    b = np.zeros((n, 8))
    b[:, 0:3] = rng.normal(size=(n, 3))
    b[:, 6] = rng.uniform(1e-9, 1e-8, n)
    b[:, 7] = rng.uniform(1e-4, 1e-3, n)
    if kind == "planar":          # zero separations on an axis, of both signs of zero
        b[:, 2] = 0.0
        b[::3, 2] = -0.0
        b[1::2, 1] = 0.25
    elif kind == "window":        # every check of the window form fails somewhere
        b[0, 0] = 1e-60           # a coordinate below 2^-140
        b[n // 2, 6] = 1e-40      # G m below 2^-100
        b[n // 3, 6] = -1e-9      # negative
        b[n // 4, 0:3] *= 1e40    # r2 above 2^190
        b[n - 1, 6] = 0.0
        b[n - 2, 0:3] = b[n - 3, 0:3] + 1e-35  # r2 far below 1
    return b


# Edges of the workgroup-per-4-bodies form (chunks of 192 bodies, wavefronts of
# 64) and operands outside the window of the branch-free quotients.
@pytest.mark.parametrize("soft", [0.0, 1e-3])
@pytest.mark.parametrize("n,kind", [(4, ""), (5, "planar"), (63, "planar"), (64, ""), (65, "window"),
                                    (191, "window"), (192, "planar"), (193, "window"),
                                    (577, "planar"), (1153, "window")])
def test_exact_bitwise_edges(ctx, n, kind, soft):
    b = _exact_edge_bodies(n, kind)
    ex = (np.random.default_rng(n).uniform(size=n) > 0.1).astype(np.int32)
    cen = (0.1, 0.2, -0.3, 1.0)
    for e in (None, ex):
        ref, rcm = orc.vector_field_brute(b, e, cen, 1.0, soft)
        acc, cm = ctx.gravity_allpairs(b, e, cen, 1.0, soft, "exact")
        on = slice(None) if e is None else e != 0
        # Coincident bodies give NaN in both; its sign is the processor's.
        a, r = acc[on], ref[on]
        assert np.all((bits(a) == bits(r)) | (np.isnan(a) & np.isnan(r)))
        assert np.array_equal(bits(cm), bits(rcm))


# Both sides of the change between the two instances of the exact kernel (8192 bodies):
# rows at the edges of chunks and workgroups, bit for bit.
@pytest.mark.parametrize("n", [8192, 8193])
def test_exact_rows_on_both_sides_of_8192(ctx, n):
    m, R = ic.disk_c3_masses(n, n)
    b = ic.disk(n, seed=n, masses=m, radii=R)
    rows = np.array([0, 3, 4, 63, 64, 191, 192, 4095, 8127, 8128, n - 2, n - 1])
    for soft in (0.0, 1e-3):
        ref = orc.vector_field_rows(b, rows, None, (1e-3, 0.0, 0.0, 1.0), 1.0, soft)
        acc, _ = ctx.gravity_allpairs(b, None, (1e-3, 0.0, 0.0, 1.0), 1.0, soft, "exact")
        assert np.array_equal(bits(acc[rows]), bits(ref))


# Massless and negative bodies are in the window: their terms' zeros and signs.
@pytest.mark.parametrize("n", [65, 193, 577])
def test_exact_massless_and_negative_bodies(ctx, n):
    b = _exact_edge_bodies(n, "planar")
    b[::3, 6] = 0.0
    b[1::6, 6] = -0.0
    b[2::3, 6] *= -1.0
    b[n // 2, 6] = 2.0 ** 100     # above the window
    cen = (0.1, 0.2, 0.0, 1.0)
    for soft in (0.0, 1e-3):
        for c in (None, cen):
            ref, rcm = orc.vector_field_brute(b, None, c, 1.0, soft)
            acc, cm = ctx.gravity_allpairs(b, None, c, 1.0, soft, "exact")
            assert np.all((bits(acc) == bits(ref)) | (np.isnan(acc) & np.isnan(ref)))
            if c is not None:
                assert np.array_equal(bits(cm), bits(rcm))
    b[:, 6] = 0.0
    ref, _ = orc.vector_field_brute(b, None, None, 1.0, 0.0)
    acc, _ = ctx.gravity_allpairs(b, None, None, 1.0, 0.0, "exact")
    assert np.array_equal(bits(acc), bits(ref))


# A flat disk with both zeros on the axis and the central body in its plane: the
# z sum of the last body at +0 is -0 (its central term, or start value, and
# every term after it), which a term of +0 for one of -0 would turn.
@pytest.mark.parametrize("n", [5, 193, 577, 1153])
def test_exact_keeps_the_sign_of_zero(ctx, n):
    b = _exact_edge_bodies(n, "flat")
    b[:, 2] = 0.0
    b[n // 4:, 2] = -0.0
    ex = (np.random.default_rng(n).uniform(size=n) > 0.1).astype(np.int32)
    ex[n // 4 - 1] = 1
    cen = (0.1, 0.2, 0.0, 1.0)
    for e in (None, ex):
        on = np.ones(n, bool) if e is None else e != 0
        ref, rcm = orc.vector_field_brute(b, e, cen, 1.0, 0.0)
        assert np.signbit(ref[n // 4 - 1, 2]) and np.all(ref[on, 2] == 0.0)
        acc, cm = ctx.gravity_allpairs(b, e, cen, 1.0, 0.0, "exact")
        assert np.array_equal(bits(acc[on]), bits(ref[on]))
        assert np.array_equal(bits(cm), bits(rcm))
        got = ctx.gravity_allpairs_from(b, central_start(b, on, cen, 1.0), e, 1.0, 0.0, "exact")
        assert np.array_equal(bits(got[on]), bits(ref[on]))


# The FP64-fast form by unordered pairs: chunks of 1024 bodies, row groups of 64
# to 512 (more rows a group above 20,000 and 65,536 bodies), remainders of every
# kind, holes at the ends; both softening kernels; the split kernel in a shape of
# the caller's gives the same to rounding (~sqrt(n) ulps of the sum; 1e-13).
@pytest.mark.parametrize("n,soft", [(4097, 0.0), (5120, 0.5), (8191, 0.0), (20001, 0.5),
                                    (65537, 0.0)])
def test_fast64_pairs_match_split_form(n, soft):
    import torch
    from ncorpion_amd import Context
    m, R = ic.disk_c3_masses(n, n)
    b = ic.disk(n, seed=n, masses=m, radii=R)
    ex = (np.random.default_rng(n).uniform(size=n) > 0.07).astype(np.int32)
    ex[[0, -1]] = 0
    cen = (1e-3, 2e-3, -1e-3, 1.0)
    bt, et = torch.from_numpy(b).cuda(), torch.from_numpy(ex).cuda()
    got = {}
    for shape in (None, (1, 32)):
        ctx = Context(0)
        try:
            if shape:
                ctx.set_tiling(shape[0], shape[1], 0.35, 0)
            for e in (None, et):
                acc = torch.full((n, 3), 7.0, dtype=torch.float64, device="cuda")
                cm = torch.zeros(3, dtype=torch.float64, device="cuda")
                torch.cuda.synchronize()
                ctx.gravity_allpairs_dev(bt, acc, e, cen, 1.0, soft, "fast64", cm)
                ctx.synchronize()
                got[shape is None, e is None] = (acc.cpu().numpy(), cm.cpu().numpy())
        finally:
            ctx.close()
    for whole in (True, False):
        (a, ca), (r, cr) = got[True, whole], got[False, whole]
        on = slice(None) if whole else ex != 0
        if not whole:
            assert np.all(a[ex == 0] == 7.0)
        assert rel_err(a[on], r[on])[1] < 1e-13
        assert np.abs(ca - cr).max() < 1e-13 * np.abs(m).sum()
    rows = np.array([1, n // 2, n - 2])
    ref = orc.vector_field_rows(b, rows, None, cen, 1.0, soft)
    ref = ref[0] if isinstance(ref, tuple) else ref
    assert rel_err(got[True, True][0][rows], ref)[0] < 1e-12


# The mixed form by unordered pairs: from 32,769 bodies, chunks of 1024, rows of
# 128 in groups of 64, more rows a group above 65,536 and 131,072; holes at the
# ends; a softening above every distance of near groups; negative and far too
# small masses.  A term's error is some six FP32 roundings (2^-24 each, half that
# in the mean), and so is the field's in the norm, at most: 1.5e-7.
@pytest.mark.parametrize("n,soft,odd", [(32769, 0.0, False), (33793, 0.5, True),
                                        (65537, 0.0, True), (131073, 0.5, False)])
def test_mixed_pairs_match_fp64(ctx, n, soft, odd):
    import torch
    m, R = ic.disk_c3_masses(n, n)
    if odd:
        m[100:230] *= -1.0
        m[5000:5003] *= 1e-40
    b = ic.disk(n, seed=n, masses=m, radii=R)
    ex = (np.random.default_rng(n).uniform(size=n) > 0.07).astype(np.int32)
    ex[[0, -1]] = 0
    cen = (1e-3, 2e-3, -1e-3, 1.0)
    bt, et = torch.from_numpy(b).cuda(), torch.from_numpy(ex).cuda()

    def field(x, e, c, prec):
        acc = torch.full((n, 3), 7.0, dtype=torch.float64, device="cuda")
        cm = torch.zeros(3, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        ctx.gravity_allpairs_dev(x, acc, e, c, 1.0, soft, prec, cm)
        ctx.synchronize()
        return acc.cpu().numpy(), cm.cpu().numpy()

    for e in (None, et):
        on = slice(None) if e is None else ex != 0
        a, _ = field(bt, e, None, "mixed")
        r, _ = field(bt, e, None, "fast64")
        if e is not None:
            assert np.all(a[ex == 0] == 7.0)
        assert np.linalg.norm(a[on] - r[on]) < 1.5e-7 * np.linalg.norm(r[on])
        (a, ca), (r, cr) = field(bt, e, cen, "mixed"), field(bt, e, cen, "fast64")
        assert np.linalg.norm(a[on] - r[on]) < 1.5e-7 * np.linalg.norm(r[on])
        assert np.abs(ca - cr).max() < 1e-13 * np.abs(m).sum()
    # Units that differ by powers of two: the same digits.
    a, _ = field(bt, None, None, "mixed")
    x = b.copy()
    x[:, 0:3] *= 2.0 ** 90
    x[:, 7] *= 2.0 ** 90
    x[:, 6] *= 2.0 ** -150
    u, _ = field(torch.from_numpy(x).cuda(), None, None, "mixed")
    assert np.array_equal(u, a * 2.0 ** -330)
    none, _ = field(bt, torch.zeros_like(et), None, "mixed")
    assert np.all(none == 7.0)


# The largest row groups (512 slots from 131,073 bodies in FP64-fast, 1024 in mixed)
# and both sides of the unordered forms' upper end (262,144): rows at every edge of
# chunks and row groups, with holes, against the oracle's sums (FP64: ~sqrt(n) ulps
# of a sum whose terms partly cancel, 1e-12; mixed: a term's FP32 rounding, 2^-24 (1 +
# 2 / theta) = 4.6e-7 at theta 0.3, twice over for a body whose terms cancel).
@pytest.mark.parametrize("n", [131073, 262144, 262145])
@pytest.mark.parametrize("prec,tol", [("fast64", 1e-12), ("mixed", 1e-6)])
def test_unordered_forms_at_their_largest(ctx, n, prec, tol):
    import torch
    m, R = ic.disk_c3_masses(n, n)
    b = ic.disk(n, seed=n, masses=m, radii=R)
    ex = (np.random.default_rng(n).uniform(size=n) > 0.07).astype(np.int32)
    rows = np.array([0, 511, 512, 1023, 1024, 65535, 131071, 131072, n - 1023, n - 2, n - 1])
    ex[rows] = 1
    bt = torch.from_numpy(b).cuda()
    for e in (None, ex):
        acc = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        et = None if e is None else torch.from_numpy(e).cuda()
        ctx.gravity_allpairs_dev(bt, acc, et, None, 1.0, 1e-6, prec)
        ctx.synchronize()
        ref = orc.vector_field_rows(b, rows, e, None, 1.0, 1e-6)
        assert rel_err(acc.cpu().numpy()[rows], ref)[0] < tol


# Without room for the partial sums of the unordered forms (here a bound of the
# caller's; an allocation that fails takes the same path) the ordered forms run:
# fields with and without holes, and graphs of RK4 steps, whose capture must not
# allocate.  FP64 sums of 1e4 terms: 1e-13; mixed against FP64 as above.
@pytest.mark.parametrize("n,prec", [(5000, "fast64"), (33000, "mixed")])
def test_fields_without_room_for_partial_sums(monkeypatch, n, prec):
    import torch
    from ncorpion_amd import Context
    m, R = ic.disk_c3_masses(n, n)
    bt = torch.from_numpy(ic.disk(n, seed=n, masses=m, radii=R)).cuda()
    et = torch.from_numpy((np.arange(n) % 11 != 3).astype(np.int32)).cuda()
    got = {}
    for room in ("", "100000"):
        monkeypatch.setenv("NCG_PAIR_SCRATCH", room)
        ctx = Context(0)
        try:
            for e in (None, et):
                acc = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
                torch.cuda.synchronize()
                ctx.gravity_allpairs_dev(bt, acc, e, None, 1.0, 0.0, prec)
                ctx.synchronize()
                got[room, e is None] = acc.cpu().numpy()
            runs = []
            for graph in (False, True):
                x = bt.clone()
                c = torch.tensor([0, 0, 0, 0, 0, 0, 1.0, 1.0], dtype=torch.float64, device="cuda")
                torch.cuda.synchronize()
                ctx.rk4_steps_dev(x, c, 4, 0.01, 1.0, 0.0, prec, graph=graph)
                ctx.synchronize()
                runs.append(x.cpu().numpy())
            assert np.array_equal(bits(runs[0]), bits(runs[1]))
        finally:
            ctx.close()
    for whole in (True, False):
        a, r = got["100000", whole], got["", whole]
        assert not np.array_equal(bits(a), bits(r))
        assert np.linalg.norm(a - r) < (1e-13 if prec == "fast64" else 1.5e-7) * np.linalg.norm(r)


# The tuning table's bound on the largest relative error (5e-7), on the disks that
# the tuner measures and the kernels that run at their sizes.
@pytest.mark.parametrize("n", [32768, 49152, 131072, 262144])
def test_mixed_error_within_the_tuners_bound(n):
    import torch
    from ncorpion_amd import Context, autotune
    bt = torch.from_numpy(autotune._workload(n)).cuda()
    acc = {p: torch.zeros((n, 3), dtype=torch.float64, device="cuda") for p in ("mixed", "fast64")}
    ctx = Context(0)
    try:
        torch.cuda.synchronize()
        for p, a in acc.items():
            ctx.gravity_allpairs_dev(bt, a, None, None, 1.0, 1e-6, p)
        ctx.synchronize()
    finally:
        ctx.close()
    assert rel_err(acc["mixed"].cpu().numpy(), acc["fast64"].cpu().numpy())[0] <= 5e-7


# theta set alone keeps the kernel (and its bits: the same theta from a table); a
# launch shape selects the split kernel.
@pytest.mark.parametrize("n,prec", [(5000, "fast64"), (33000, "mixed")])
def test_theta_alone_keeps_the_unordered_form(monkeypatch, tmp_path, n, prec):
    import torch
    from ncorpion_amd import Context
    table = tmp_path / "tuning.txt"
    table.write_text("mixed 1 1 0 0.45 0\nfast64 1 1 0 0.45 0\n")
    monkeypatch.setenv("NCG_TUNING", str(table))
    m, R = ic.disk_c3_masses(n, n)
    bt = torch.from_numpy(ic.disk(n, seed=n, masses=m, radii=R)).cuda()
    got = []
    for args in (None, dict(theta=0.45), dict(ipl=1, theta=0.45)):
        ctx = Context(0)
        try:
            if args:
                ctx.set_tiling(**args)
            acc = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            ctx.gravity_allpairs_dev(bt, acc, None, None, 1.0, 0.0, prec)
            ctx.synchronize()
            got.append(acc.cpu().numpy())
        finally:
            ctx.close()
    assert np.array_equal(bits(got[0]), bits(got[1]))
    assert not np.array_equal(bits(got[0]), bits(got[2]))


# Softening beyond the system: every pair of groups is near, the far kernel forms
# nothing and its sums (an earlier call's) are left out.  FP64 sums of 3e4 terms:
# ~sqrt(n) ulps, 1e-13.
@pytest.mark.parametrize("n", [32769, 40001])
def test_mixed_pairs_all_near(ctx, n):
    import torch
    m, R = ic.disk_c3_masses(n, n)
    bt = torch.from_numpy(ic.disk(n, seed=n, masses=m, radii=R)).cuda()

    def field(soft, prec):
        acc = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        ctx.gravity_allpairs_dev(bt, acc, None, None, 1.0, soft, prec)
        ctx.synchronize()
        return acc.cpu().numpy()

    far = field(0.0, "mixed")
    near, ref = field(10.0, "mixed"), field(10.0, "fast64")
    assert np.linalg.norm(near - ref) < 1e-13 * np.linalg.norm(ref)
    assert np.array_equal(field(0.0, "mixed"), far)
