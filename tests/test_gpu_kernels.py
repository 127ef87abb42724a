"""Kernels at the sizes where their tilings can go wrong (remainders, the
smallest and largest of a range), each against the CPU oracle."""
import numpy as np
import pytest

from test_gpu_parity import assert_close, interior, make_pair, pinned_gauge  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jtot", [8, 60, 64, 512, 540, 2048, 2250])
def test_diagnostics_partial_counts(sns, jtot):
    """The last reduction of the monitors over few slots, one full round of
    its threads (64 slots), whole and ragged unrolled rounds (512, 540) and
    the most slots (2048; 2250 rows share them): sums of jtot*itot terms of
    one sign to 1e-12, as the sequential ones."""
    o, inst = make_pair(sns, 8, jtot, 3.0, seed=jtot)
    d = inst.diagnostics()
    ene, nu = o.energy(), o.nusselt()
    assert d["divmax"] == o.divergence()[0]
    for k, ref in (("energy_ux", ene[0]), ("energy_uy", ene[1]), ("energy_t", ene[2]),
                   ("nu_eps_k", nu[2]), ("nu_eps_h", nu[3])):
        assert abs(d[k] - ref) <= 1e-12 * abs(ref), (k, d[k], ref)
    inst.close()


# (itot, jtot, dt, Ra): chunk lengths 4 to 32 (every register tile of the
# kernel and its remainders), 4 to 256 chunks, 4 to 16 columns per workgroup
# with ragged last tiles; lambda = pf/dy^2 from 1e-4 (no doubling step) to
# 1e3 (the sums wrap around the period many times)
YCOL_CASES = [
    (8, 16, 1e-3, 1e8), (5, 16, 1.0, 1e2), (33, 45, 1e-2, 1e6), (19, 96, 1.0, 1e2),
    (37, 200, 0.1, 1e4), (17, 324, 1e-2, 1e8), (12, 1000, 0.1, 1e4), (40, 960, 1e-3, 1e8),
    (70, 2048, 1e-2, 1e6), (21, 4096, 1e-3, 1e6), (13, 8192, 1e-3, 1e4),
]


@pytest.mark.parametrize("case", YCOL_CASES)
def test_ycol_against_oracle(sns, case):
    """Crank-Nicolson in y by whole columns, T and both velocities, against
    the oracle's sequential periodic sweeps.  The diagonal 1 + 2 lambda is
    rounded to eps (1 + 2 lambda) while the smallest eigenvalue is 1, so two
    correct solvers differ by a few eps (1 + 2 lambda)."""
    itot, jtot, dt, Ra = case
    o, inst = make_pair(sns, itot, jtot, 3.0, 0, 1, seed=31, dt=dt, Ra=Ra)
    lam = 0.5 * dt * max(2.0 ** -0.5, 2.0 ** 0.5) / Ra ** 0.5 * (jtot / 2.0) ** 2
    tol = 1e-13 + 32 * np.finfo(float).eps * (1 + 2 * lam)
    o.update_temp(1)
    inst.update_temp(1)
    o.update_velocity(1)
    inst.update_velocity(1)
    for n in ("temp", "ux", "uy"):
        assert_close(inst.download(n)[1:-1], o.f[n][1:-1], tol, n)
    inst.close()


@pytest.mark.parametrize("itot", [4, 63, 64, 65, 256, 257, 512, 513, 1024, 1025, 2049, 4097])
def test_x_solves_at_row_widths(sns, pinned_gauge, itot):  # noqa: F811
    """The affine scans of the x solves at one lane, one wave and the edges of
    every row width (threads x unknowns per thread): the implicit-x update of
    T to the bar of the sequential sweep (1e-13) and the potential to 1e-11
    after removing its mean, as the other sizes are held to."""
    o, inst = make_pair(sns, itot, 8, float(itot), 1, 0, seed=itot)
    o.update_temp(1)
    inst.update_temp(1)
    assert_close(inst.download("temp"), o.f["temp"], 1e-13, "temp")
    o.compute_potential(1)
    inst.compute_potential(1)
    assert_close(interior(inst.download("psi")), interior(o.f["psi"]), 1e-11, "psi", demean=True)
    inst.close()


# itot at the edges of the stencil blocks (124 columns, the ux pairs one
# column early) and of the rows' shapes (2, 4 and 8 unknowns per thread, by the
# number of rows), odd row counts, one wave to sixteen
ROW_CASES = [(4, 4), (5, 9), (123, 12), (124, 15), (125, 12), (126, 8), (248, 12), (249, 8),
             (250, 8), (373, 1440), (512, 1024), (512, 2700), (1024, 16), (1025, 8), (4097, 6),
             (8192, 4)]


@pytest.mark.parametrize("imy", [0, 1])
@pytest.mark.parametrize("itot,jtot", ROW_CASES)
def test_row_predictor_edges(sns, itot, jtot, imy):
    """Two fused steps (the corrections folded into the predictor with
    explicit y) against the reference-named functions, whose source terms
    equal the oracle's bit for bit: every field equal, stretched grid."""
    if imy and jtot < 16:
        jtot = 16
    fields = {}
    for fused in (False, True):
        inst = sns.Instance(itot, jtot, stretch=3.0, Ra=1e7, Pr=2.0, implicitx=1, implicity=imy)
        inst.alloc()
        inst.state_alloc()
        rng = np.random.default_rng(itot + jtot)
        for n in ("ux", "uy", "p", "temp"):
            inst.upload(n, 0.1 * rng.standard_normal(inst.shape(n)))
            inst.update_boundaries(n)
            inst.state_upload(n, inst.download(n))
        inst.set_dt(1e-4)
        for _ in range(2):
            inst.integrate() if fused else inst.integrate_reference_order()
        for n in ("ux", "uy", "p", "temp"):
            inst.update_boundaries(n)
            got = inst.state_download(n) if fused else inst.download(n)
            assert np.isfinite(got).all()
            if fused:
                assert np.array_equal(got, fields[n]), (n, np.abs(got - fields[n]).max())
            fields[n] = got
        inst.close()


# itot at the edges of the blocks (124 columns) and of the workgroups (four
# blocks), odd row counts; stretch 0 is the Chebyshev grid
EXP_CASES = [(4, 4, 0.), (5, 9, 3.), (64, 64, 0.), (123, 12, 3.), (124, 15, 0.), (125, 12, 3.),
             (128, 192, 0.), (248, 9, 3.), (249, 8, 0.), (497, 12, 3.), (512, 32, 0.),
             (1024, 15, 0.)]


@pytest.mark.parametrize("imy", [0, 1])
@pytest.mark.parametrize("with_t", [1, 0])
@pytest.mark.parametrize("itot,jtot,stretch", EXP_CASES)
def test_explicit_x_predictor_edges(sns, itot, jtot, stretch, with_t, imy):
    """Explicit diffusion in x: two fused steps (the corrections folded into
    the predictor with explicit y) against the reference-named functions:
    every field equal."""
    if imy and jtot < 16:
        jtot = 16
    fields = {}
    for fused in (False, True):
        inst = sns.Instance(itot, jtot, stretch=stretch, Ra=1e7, Pr=2.0, implicitx=0,
                            implicity=imy, with_temperature=with_t)
        inst.alloc()
        inst.state_alloc()
        rng = np.random.default_rng(itot + jtot)
        for n in ("ux", "uy", "p", "temp"):
            inst.upload(n, 0.1 * rng.standard_normal(inst.shape(n)))
            inst.update_boundaries(n)
            inst.state_upload(n, inst.download(n))
        inst.set_dt(1e-6)
        for _ in range(2):
            inst.integrate() if fused else inst.integrate_reference_order()
        for n in ("ux", "uy", "p", "temp"):
            inst.update_boundaries(n)
            got = inst.state_download(n) if fused else inst.download(n)
            assert np.isfinite(got).all()
            if fused:
                assert np.array_equal(got, fields[n]), (n, np.abs(got - fields[n]).max())
            fields[n] = got
        inst.close()


# (itot, jtot, first factor of the two passes or 0 for the rule): whole columns in
# one kernel up to 1024 rows with 1, 2 and 4 column pairs a workgroup (compiled
# and read schedules, one stage, odd lengths), two passes above (two and three
# stages, factors of 16*16 and 3*9*9, a half tile of columns)
FFT_CASES = [(4, 4, 0), (5, 6, 0), (4, 10, 0), (16, 16, 0), (31, 32, 0), (33, 75, 0), (255, 64, 0),
             (256, 48, 0), (17, 192, 0), (257, 1000, 0), (40, 243, 0), (1023, 128, 0),
             (1024, 320, 0), (1025, 1024, 0), (16, 1080, 0), (17, 1125, 0), (9, 2048, 0),
             (40, 2000, 0), (5, 1458, 0), (33, 486, 243), (7, 512, 256), (18, 250, 125),
             (6, 16384, 0)]


@pytest.mark.parametrize("itot,jtot,n1", FFT_CASES)
def test_transforms_by_length(sns, pinned_gauge, itot, jtot, n1):  # noqa: F811
    """The potential to 1e-11 of the oracle's after removing its mean (the bar
    of the other sizes), and two fused steps (padded layout) equal to the
    reference-named functions (packed layout)."""
    o, inst = make_pair(sns, itot, jtot, 3.0, 0, 0, seed=itot + jtot)
    inst.set_launch(fft_n1=n1)
    assert inst.launch()["fft_n1"] == n1 or jtot > 1024
    o.compute_potential(1)
    inst.compute_potential(1)
    assert_close(interior(inst.download("psi")), interior(o.f["psi"]), 1e-11, "psi", demean=True)
    names = ("ux", "uy", "p", "temp")
    inst.state_alloc()
    for n in names:
        inst.update_boundaries(n)
        inst.state_upload(n, inst.download(n))
    inst.set_dt(1e-8)
    for _ in range(2):  # T's two buffers: back in the one that holds the corners
        inst.integrate()
        inst.integrate_reference_order()
    for n in names:
        inst.update_boundaries(n)
        assert np.array_equal(inst.state_download(n), inst.download(n)), n
    inst.close()


# (itot, jtot, implicit x, y): partial minima at the edges of the rule (512 for
# the explicit predictor, 2048 for the factors) and a few
DT_CASES = [(4, 8, 0, 0), (248, 1024, 0, 0), (249, 1024, 0, 0), (248, 1024, 0, 1),
            (16, 4096, 0, 1), (16, 4320, 0, 1), (16, 4096, 1, 0), (16, 4320, 1, 0),
            (300, 24, 1, 1)]


@pytest.mark.parametrize("itot,jtot,imx,imy", DT_CASES)
def test_time_step_decided_by_first_kernel(sns, itot, jtot, imx, imy):
    """Three steps of the time loop, whose first kernels decide dt, against
    dt decided on the host before each step: dt, time and fields equal."""
    def make():
        inst = sns.Instance(itot, jtot, stretch=3.0, Ra=1e6, Pr=2.0, implicitx=imx, implicity=imy)
        inst.state_alloc()
        inst.state_init_temperature(itot + jtot, 1e-2)
        return inst
    a, b = make(), make()
    a.advance(3)
    t = 0.0
    for _ in range(3):
        dt = sns.decide_dt(b.g, 1e6, 2.0, b.state_dt_adv_raw(), imx, imy)
        b.set_dt(dt)
        b.integrate()
        t += dt
    assert a.get_time() == (t, dt)
    for n in ("ux", "uy", "p", "temp"):
        assert np.array_equal(a.state_download(n), b.state_download(n)), n
    a.close()
    b.close()


# one field in one piece, and in several with a ragged last one (8 MiB pieces)
@pytest.mark.parametrize("itot,jtot", [(4, 4), (33, 75), (700, 1620), (8192, 270)])
def test_state_fields_to_and_from_the_host(sns, itot, jtot):
    """Every value of an uploaded field comes back, and the padding of the
    device rows is not part of it."""
    inst = sns.Instance(itot, jtot)
    inst.state_alloc()
    rng = np.random.default_rng(itot)
    for n in ("ux", "uy", "p", "temp"):
        a = rng.standard_normal(inst.shape(n))
        inst.state_upload(n, a)
        assert np.array_equal(inst.state_download(n), a), n
    inst.close()


def test_state_copies_need_no_state_of_the_instance(sns):
    """The rows that state copies go through are the instance's from the start:
    an instance without a state of its own copies the state of another one of
    its grid, and freeing a state gives back what allocating it took."""
    a, b = sns.Instance(40, 60), sns.Instance(40, 60)
    before = a.memory(), b.memory()
    a.state_alloc()
    taken = a.memory() - before[0]
    b.state_alloc()
    assert b.L.snsg_state_free(b.ctx, b.state) == 0
    assert taken > 0 and b.memory() == before[1]
    b.state = a.state
    f = np.random.default_rng(1).standard_normal(a.shape("ux"))
    b.state_upload("ux", f)
    assert np.array_equal(b.state_download("ux"), f)
    assert np.array_equal(a.state_download("ux"), f)
    b.state = None
    a.close()
    b.close()


# (itot, jtot, stretch, correction kernels in a step): the widest rows that fold
# with the division sequence, the first and the widest that do not, and a wide
# one that divides by multiplying
FOLD_RULE_CASES = [(2048, 9, 3., 1), (2049, 9, 3., 3), (2049, 1024, 3., 3), (8192, 8, 3., 3),
                   (4096, 8, 4096., 1), (4097, 8, 4097., 3)]


@pytest.mark.parametrize("itot,jtot,stretch,ncorr", FOLD_RULE_CASES)
def test_fold_rule_of_wide_rows(sns, itot, jtot, stretch, ncorr):
    """With implicit x the correction is folded into the predictor except where
    its division sequence would spill registers; the fields are those of the
    sequence with the correction kernel either way."""
    out = []
    for split in (0, 1):
        inst = sns.Instance(itot, jtot, stretch=stretch, Ra=1e8, Pr=0.7, implicitx=1, implicity=0)
        inst.set_launch(split_corr=split)
        inst.state_alloc()
        rng = np.random.default_rng(itot + jtot)
        for n in ("ux", "uy", "p", "temp"):
            inst.state_upload(n, 1e-3 * rng.standard_normal(inst.shape(n)))
        inst.set_dt(1e-6)
        inst.timing_enable("corr")
        inst.integrate()
        assert inst.timing_read()[0] == (3 if split else ncorr)
        inst.timing_disable()
        inst.advance(2)
        out.append({n: inst.state_download(n) for n in ("ux", "uy", "p", "psi", "temp")})
        inst.close()
    for n in out[0]:
        assert np.array_equal(out[0][n], out[1][n]), n


def test_batch_of_wide_rows_mixes_divisors(sns):
    """A wide uniform member with powers of two for divisors and a stretched
    one in one class: neither folds, both end where they end alone."""
    def make(stretch):
        inst = sns.Instance(4096, 8, stretch=stretch, Ra=1e8, Pr=0.7, implicitx=1, implicity=0)
        inst.state_alloc()
        inst.state_init_temperature(3, 1e-2)
        return inst
    insts, refs = [make(4096.), make(3.)], [make(4096.), make(3.)]
    batch = sns.Batch(insts)
    assert batch.classes() == 1
    batch.advance(3)
    for r in refs:
        r.advance(3)
    batch.sync()
    for i, r in zip(insts, refs):
        for n in ("ux", "uy", "p", "psi", "temp"):
            assert np.array_equal(i.state_download(n), r.state_download(n)), n
        assert i.get_time() == r.get_time()
    batch.close()
    for i in insts + refs:
        i.close()


# (itot, jtot, first factor of the two passes or 0 for the rule, stretch): every
# pair of compiled schedules (factors of 32, 64 and 128), whole and half tiles
TWO_PASS_CASES = [(9, 2048, 0, 3.), (16, 2048, 0, 16.), (12, 4096, 0, 3.), (16, 4096, 0, 16.),
                  (20, 8192, 0, 3.), (8, 8192, 128, 8.), (7, 16384, 0, 3.), (33, 1024, 32, 3.)]


@pytest.mark.parametrize("itot,jtot,n1,stretch", TWO_PASS_CASES)
def test_two_pass_schedules_on_both_layouts(sns, pinned_gauge, itot, jtot, n1, stretch):  # noqa: F811
    """The two passes with compiled schedules: psi on the packed layout to 1e-11
    of the oracle's after removing its mean (the bar of the other lengths),
    and the padded layout's after one fused step equal to it bit for bit."""
    o, inst = make_pair(sns, itot, jtot, stretch, 0, 0, seed=itot + jtot)
    inst.set_launch(fft_n1=n1)
    assert inst.launch()["fft_n1"] >= 32
    o.compute_potential(1)
    inst.compute_potential(1)
    assert_close(interior(inst.download("psi")), interior(o.f["psi"]), 1e-11, "psi", demean=True)
    inst.state_alloc()
    for n in ("ux", "uy", "p", "temp"):
        inst.update_boundaries(n)
        inst.state_upload(n, inst.download(n))
    inst.set_dt(1e-8)
    inst.integrate()
    inst.integrate_reference_order()
    assert np.array_equal(inst.state_download("psi"), inst.download("psi"))
    inst.close()


# Uniform grids: powers of two for every divisor (the kernels multiply), uniform
# spacings in x with another dy (they divide, with the spacings of interior
# blocks as constants), and widths whose uniform spacings differ in their last
# bits (they divide by the tables'); one block to many, one to several workgroups
# per row
UNIFORM_CASES = [(4, 4, True), (64, 64, True), (128, 16, True), (256, 8, True), (512, 32, True),
                 (512, 2048, True), (1024, 16, True), (2048, 8, True), (4096, 8, True),
                 (8192, 4, True), (128, 15, False), (256, 90, False), (512, 45, False),
                 (1024, 1080, False), (2048, 12, False), (4096, 9, False), (250, 8, False),
                 (373, 12, False), (500, 15, False), (1000, 16, False), (3000, 9, False)]


@pytest.mark.parametrize("imx,imy", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("itot,jtot,pow2", UNIFORM_CASES)
def test_predictors_on_uniform_grids(sns, itot, jtot, pow2, imx, imy):
    """Two fused steps against the reference-named functions, whose source
    terms equal the oracle's bit for bit: every field equal."""
    if imy and jtot < 16:
        jtot = 16 if pow2 else 18
    fields = {}
    for fused in (False, True):
        inst = sns.Instance(itot, jtot, stretch=float(itot), Ra=1e7, Pr=2.0, implicitx=imx,
                            implicity=imy)
        assert inst.uniform_grid() == (itot & (itot - 1) == 0)
        spacings = list(inst.g["dxf"]) + list(inst.g["dxc"]) + [2.0 / jtot]
        assert all(np.frexp(v)[0] == 0.5 for v in spacings) == pow2
        inst.alloc()
        inst.state_alloc()
        rng = np.random.default_rng(itot + jtot)
        for n in ("ux", "uy", "p", "temp"):
            inst.upload(n, 0.1 * rng.standard_normal(inst.shape(n)))
            inst.update_boundaries(n)
            inst.state_upload(n, inst.download(n))
        inst.set_dt(1e-7)
        for _ in range(2):
            inst.integrate() if fused else inst.integrate_reference_order()
        for n in ("ux", "uy", "p", "temp"):
            inst.update_boundaries(n)
            got = inst.state_download(n) if fused else inst.download(n)
            assert np.isfinite(got).all()
            if fused:
                assert np.array_equal(got, fields[n]), (n, np.abs(got - fields[n]).max())
            fields[n] = got
        inst.close()
