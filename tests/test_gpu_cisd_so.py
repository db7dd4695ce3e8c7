"""GPU parity of the spin-orbital CISD / CID path against the oracle."""
import numpy as np
import pytest
import torch

from apyib_amd import synthetic
from apyib_amd.so_ci import SOCI, SOIntegrals, npair, so_fock_from_mo
from oracle import brute, so, transforms
from tests.gpu_layouts import expected_blocks
from tests.helpers import PARAMS, brillouin, rand_amplitudes

pytestmark = pytest.mark.gpu

SIZES = [(4, 6, 3), (6, 8, 5), (5, 7, 9), (2, 3, 1)]


def _dev(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


@pytest.mark.parametrize("O,V,seed", SIZES)
def test_synthetic_blocks_match_host_generator(dev, O, V, seed):
    A = synthetic.eri_full(O + V, seed)
    exp = expected_blocks(A, O)
    ints = SOIntegrals.synthetic(O, V, seed, device=dev)
    for name, want in exp.items():
        got = ints[name].cpu().numpy()
        assert np.abs(got - want).max() < 1e-15, name


@pytest.mark.parametrize("O,V,seed", SIZES)
def test_blocks_from_full_are_exact_copies(dev, O, V, seed):
    A = synthetic.eri_full(O + V, seed)
    ints = SOIntegrals.from_full(_dev(A, dev), O)
    for name, want in expected_blocks(A, O).items():
        assert np.array_equal(ints[name].cpu().numpy(), want), name


@pytest.mark.parametrize("m,Osp", [(5, 4), (6, 6), (4, 2)])
def test_blocks_from_mo_spin_expansion(dev, m, Osp):
    rng = np.random.default_rng(m)
    eri_mo = rng.standard_normal((m,) * 4) + 1j * rng.standard_normal((m,) * 4)
    eri_so = transforms.compute_ERI_SO(eri_mo).swapaxes(1, 2)        # Dirac <pq|rs>
    A = eri_so - eri_so.swapaxes(2, 3)                                 # <pq||rs> per term
    ints = SOIntegrals.from_mo(_dev(eri_mo, dev), Osp)
    for name, want in expected_blocks(A, Osp).items():
        assert np.abs(ints[name].cpu().numpy() - want).max() < 1e-14, name
    f_mo = rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))
    f_so = so_fock_from_mo(_dev(f_mo, dev)).cpu().numpy()
    assert np.array_equal(f_so, transforms.compute_F_SO_loop(f_mo))


@pytest.mark.parametrize("m,Osp", [(2, 1), (33, 3), (40, 7), (70, 4), (36, 70), (44, 19), (48, 22), (65, 71)])
def test_blocks_from_mo_at_tile_edges(dev, m, Osp):
    """The spin-expanded blocks of apy_so_ints_from_mo against those of apy_so_ints_from_full (the general
    element-wise path) on the expanded tensor: virtual spaces below, at and past one and two 32-wide spatial
    tiles, an odd number of occupied spin orbitals, more than 32 occupied spatial orbitals, each block on
    either side of the size from which its rows are built by spatial pairs.  Copies and single differences:
    equal."""
    n = 2 * m
    g = torch.Generator(device=dev).manual_seed(m)
    E = torch.randn((m,) * 4, dtype=torch.complex128, device=dev, generator=g)
    if n > 80:                       # the expanded tensor of 80 spin orbitals is 0.7 GB: larger ones by blocks
        names = ("ring", "vovv_p", "vvvo_p")
        got = SOIntegrals.from_mo(E, Osp, blocks=names)
        V = n - Osp
        o, v = torch.arange(Osp, device=dev), Osp + torch.arange(V, device=dev)
        a, b = torch.triu_indices(V, V, 1, device=dev) + Osp

        def anti(p, q, r, s):
            z = torch.zeros((), dtype=torch.complex128, device=dev)
            d = torch.where(((p ^ r) & 1 == 0) & ((q ^ s) & 1 == 0), E[p >> 1, r >> 1, q >> 1, s >> 1], z)
            return d - torch.where(((p ^ s) & 1 == 0) & ((q ^ r) & 1 == 0), E[p >> 1, s >> 1, q >> 1, r >> 1], z)

        ring = torch.stack([anti(o[None, :, None], v[:, None, None], v[None, None, :], j) for j in o])
        assert torch.equal(got["ring"], ring.reshape(-1))
        vovv = got["vovv_p"].view(V, Osp, -1)
        vvvo = got["vvvo_p"].view(-1, Osp, V)
        for k in range(0, V, 7):
            assert torch.equal(vovv[k], anti(v[k], o[:, None], a[None], b[None]))
        for k in range(0, a.numel(), 997):
            assert torch.equal(vvvo[k], anti(a[k], b[k], v[None], o[:, None]))
        return
    p = torch.arange(n, device=dev)
    same = (p[:, None] & 1) == (p[None, :] & 1)
    h = p >> 1
    D = E[h][:, h][:, :, h][:, :, :, h] * (same[:, :, None, None] & same[None, None])     # (pr|qs) spin-expanded
    A = D.permute(0, 2, 1, 3) - D.permute(0, 2, 3, 1)                                     # <pq||rs>
    got, want = SOIntegrals.from_mo(E, Osp), SOIntegrals.from_full(A, Osp)
    for name in want.blocks:
        assert torch.equal(got[name], want[name]), name


def test_small_blocks_stay_in_the_caches(dev):
    """Blocks that fit the caches are read from them after they are built: building and reading those of 16
    orbitals took a third longer when every block was stored past the caches."""
    m, O = 16, 10
    E = torch.randn((m,) * 4, dtype=torch.complex128, device=dev)
    blocks = SOIntegrals.from_mo(E, O)
    flat = [blocks[name].view(torch.float64) for name in blocks.blocks]
    into = [torch.empty_like(x) for x in flat]

    def us(build):
        best = float("inf")
        for _ in range(20):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            build()
            a.record()
            for x, y in zip(flat, into):
                torch.sum(x, dim=0, out=y[:1].squeeze(0))
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    def rebuild():
        import ctypes
        from apyib_amd import _lib
        from apyib_amd.kernels import stream_of
        _lib.check(_lib.load().apy_so_ints_from_mo(m, ctypes.c_void_p(E.data_ptr()), ctypes.byref(blocks.struct),
                                                   stream_of(dev)), "apy_so_ints_from_mo")

    def fill():
        for x in flat:
            x.zero_()

    assert us(rebuild) < 1.15 * us(fill)


@pytest.mark.parametrize("O,V", [(2, 2), (3, 5), (5, 33), (10, 4), (9, 64), (13, 41)])
@pytest.mark.parametrize("singles,fov,fold,packed", [(True, False, True, False), (True, True, True, True),
                                                     (True, True, False, False), (False, False, True, False)])
def test_grouped_products_match_one_after_another(dev, O, V, singles, fov, fold, packed):
    """A step's products in one launch against the same products one launch after another (the form that timing
    events ask for; they time the first product, so both must have been recorded): two orders of sums of up to
    O V^2 terms of order one.  The products share targets (R and the singles) and, at the larger sizes, have several
    K slices each."""
    import ctypes
    from apyib_amd import _lib
    lib = _lib.load()
    F, eps = synthetic.fock(O, V, 3)
    ints = SOIntegrals.synthetic(O, V, 3, device=dev)
    ci = SOCI(ints, _dev(F, dev), eps, singles=singles, fov_coupling=fov, fold_fvv=fold)
    g = torch.Generator(device=dev).manual_seed(O * V)
    t = torch.randn(ci.Lp if packed else ci.L, dtype=torch.complex128, device=dev, generator=g) * 0.1
    mode = _lib.APY_MODE_SIGMA if packed or fov else _lib.APY_MODE_RESIDUAL

    def run(events):
        out, tn = torch.full_like(t, 7.0), torch.full_like(t, 7.0)
        ev = [e.cuda_event for e in events] if events else [None, None]
        a = _lib.CisdSoArgs(O, V, ci.fock.data_ptr(), ci.eps.data_ptr(), ctypes.pointer(ints.struct), ci.hoo.data_ptr(),
                            int(singles), int(mode), int(fov), ci.energy_dev.data_ptr(), 1.0, 0.0, t.data_ptr(),
                            tn.data_ptr(), out.data_ptr(), *ev, None,
                            ci.ring_f.data_ptr() if fold else None, int(packed), 0)
        ws = torch.empty(ci.ws_bytes, dtype=torch.uint8, device=dev)
        assert lib.apy_cisd_so_step(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), ci.ws_bytes,
                                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        torch.cuda.synchronize()
        return out, tn

    grouped = run(None)
    events = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    for e in events:
        e.record()                                      # creates the handles
    torch.cuda.synchronize()
    alone = run(events)
    assert 0.0 < events[0].elapsed_time(events[1]) < 1e3
    if O * V > 500:                                     # other tiles and slices: not the same sums bit for bit
        assert not torch.equal(grouped[0], alone[0])
    live = slice(None) if singles else slice(ci.OV, None)
    for x, y in zip(grouped, alone):
        assert (x[live] - y[live]).abs().max() <= 1e-13 * max(1.0, y[live].abs().max().item())


@pytest.mark.parametrize("O,V", [(2, 9), (4, 20), (6, 40), (8, 33), (11, 21), (12, 30)])
@pytest.mark.parametrize("packed", [False, True])
def test_three_product_form_by_rows(dev, O, V, packed):
    """The three-product option against the four products where the ladder has few rows (it keeps four products
    on a narrower tile there) and where it has enough; sums of up to V^2 / 2 terms of order one, and the
    three-product form's two differences of them."""
    F, eps = synthetic.fock(O, V, 5)
    ints = SOIntegrals.synthetic(O, V, 5, device=dev)
    ci = SOCI(ints, _dev(F, dev), eps, fov_coupling=True)
    g = torch.Generator(device=dev).manual_seed(V)
    x = torch.randn(ci.Lp if packed else ci.L, dtype=torch.complex128, device=dev, generator=g)
    a, b = torch.zeros_like(x), torch.zeros_like(x)
    ci.sigma(x, a, packed=packed)
    ci.gauss3m = True
    ci.sigma(x, b, packed=packed)
    assert (a - b).abs().max() <= 1e-13 * a.abs().max()


def test_three_product_form_of_few_rows_is_no_slower(dev):
    """Six rows on a 64-row tile cost ten times their products: the three-product option took twice the time of
    the four products it is meant to save."""
    O, V = 4, 150
    F, eps = synthetic.fock(O, V, 5)
    ci = SOCI(SOIntegrals.synthetic(O, V, 5, device=dev), _dev(F, dev), eps, fov_coupling=True)
    x, y = ci.new_vector(), ci.new_vector()

    def us():
        best = float("inf")
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ci.sigma(x, y)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    four = us()
    ci.gauss3m = True
    assert us() < 1.3 * four


def _system(O, V, seed, dev, brill=False):
    F, A, eps = synthetic.system(O, V, seed)
    if brill:
        F = brillouin(F, O)
    ints = SOIntegrals.synthetic(O, V, seed, device=dev)
    return F, A, eps, ints


@pytest.mark.parametrize("O,V,seed", SIZES)
@pytest.mark.parametrize("singles", [True, False])
def test_residual_step_matches_oracle(dev, O, V, seed, singles):
    F, A, eps, ints = _system(O, V, seed, dev)
    t1, t2 = rand_amplitudes(O, V, seed + 1)
    if not singles:
        t1 = np.zeros_like(t1)
    E = 0.013 - 0.002j
    solver = SOCI(ints, _dev(F, dev), eps, singles=singles)
    t = _dev(np.concatenate([t1.ravel(), t2.ravel()]), dev)
    tn = solver.new_vector()
    r = solver.new_vector()
    Ed = torch.tensor([E], dtype=torch.complex128, device=dev)
    solver.step(t, tn, r, energy=Ed)
    D1, D2 = so.denominators(eps[:O], eps[O:])
    if singles:
        r1, r2 = so.cisd_so_residual(F, A / 2, t1, t2, E, O)
    else:
        r1, r2 = np.zeros_like(t1), so.cid_so_residual(F, A / 2, t2, E, O)
    g1, g2 = solver.split(r)
    n1, n2 = solver.split(tn)
    scale = max(1.0, np.abs(r2).max())
    assert np.abs(g2.cpu().numpy() - r2).max() < 1e-13 * scale
    assert np.abs(n2.cpu().numpy() - (t2 + r2 / D2)).max() < 1e-12
    if singles:
        assert np.abs(g1.cpu().numpy() - r1).max() < 1e-13 * scale
        assert np.abs(n1.cpu().numpy() - (t1 + r1 / D1)).max() < 1e-12


@pytest.mark.parametrize("O,V,seed", [(4, 5, 3), (2, 4, 5)])
def test_sigma_mode_hermitian_matches_determinant_ci(dev, O, V, seed):
    """sigma(c0, x) with the f_vo coupling switched on is the CI matrix-vector
    product, including the reference weight c0."""
    F, A, eps, ints = _system(O, V, seed, dev)
    t1, t2 = rand_amplitudes(O, V, seed + 3)
    c0 = 0.7 - 0.2j
    n = O + V
    sp = brute.CISpace(n, O)
    H, Eref = brute.hamiltonian(F, A, sp)
    c = brute.vector_from_amplitudes(sp, t1, t2, c0=c0)
    _, s1, s2 = brute.amplitudes_from_vector(sp, H @ c - Eref * c, V)
    solver = SOCI(ints, _dev(F, dev), eps, singles=True, fov_coupling=True)
    x = _dev(np.concatenate([t1.ravel(), t2.ravel()]), dev)
    out = solver.new_vector()
    solver.sigma(x, out, c0=c0)
    g1, g2 = solver.split(out)
    assert np.abs(g1.cpu().numpy() - s1).max() < 1e-13
    assert np.abs(g2.cpu().numpy() - s2).max() < 1e-13


@pytest.mark.parametrize("O,V,seed", [(4, 6, 3), (6, 8, 5), (2, 5, 2)])
def test_solve_cisd_so_matches_oracle(dev, O, V, seed):
    F, A, eps, ints = _system(O, V, seed, dev)
    E_ref, t1_ref, t2_ref, it_ref = so.solve_cisd_so(F, A / 2, eps[:O], eps[O:], O, PARAMS)
    solver = SOCI(ints, _dev(F, dev), eps, singles=True)
    E, t1, t2, it = solver.solve(PARAMS)
    assert abs(E - E_ref) < 1e-10
    assert np.abs(t1.cpu().numpy() - t1_ref).max() < 1e-9
    assert np.abs(t2.cpu().numpy() - t2_ref).max() < 1e-9
    assert abs(it - it_ref) <= 1


@pytest.mark.parametrize("O,V,seed", [(4, 6, 3), (6, 7, 1)])
def test_solve_cid_so_matches_oracle(dev, O, V, seed):
    F, A, eps, ints = _system(O, V, seed, dev)
    E_ref, t2_ref, it_ref = so.solve_cid_so(F, A / 2, eps[:O], eps[O:], O, PARAMS)
    solver = SOCI(ints, _dev(F, dev), eps, singles=False)
    E, _, t2, it = solver.solve(PARAMS)
    assert abs(E - E_ref) < 1e-10
    assert np.abs(t2.cpu().numpy() - t2_ref).max() < 1e-9


def test_solve_without_diis_matches_oracle(dev):
    O, V, seed = 4, 6, 4
    F, A, eps, ints = _system(O, V, seed, dev)
    p = dict(PARAMS, DIIS=False, max_iterations=400)
    E_ref, t1_ref, t2_ref, _ = so.solve_cisd_so(F, A / 2, eps[:O], eps[O:], O, p)
    E, t1, t2, _ = SOCI(ints, _dev(F, dev), eps).solve(p)
    assert abs(E - E_ref) < 1e-10
    assert np.abs(t2.cpu().numpy() - t2_ref).max() < 1e-9


def test_max_iterations_reached_returns_last_iterate(dev, capsys):
    O, V, seed = 4, 6, 4
    F, A, eps, ints = _system(O, V, seed, dev)
    p = dict(PARAMS, max_iterations=2)
    E_ref, _, t2_ref, _ = so.solve_cisd_so(F, A / 2, eps[:O], eps[O:], O, p)
    E, _, t2, it = SOCI(ints, _dev(F, dev), eps).solve(p)
    assert it == 2
    assert abs(E - E_ref) < 1e-12
    assert "Not converged." in capsys.readouterr().out


# virtual spaces wider than one 32-wide epilogue tile (several tile pairs, a
# ragged last tile) and the narrowest case
WIDE = [(4, 40, 3), (3, 45, 7), (2, 33, 2), (2, 2, 4)]


def _packed(t1, t2, O, V, extra=()):
    io, jo = np.triu_indices(O, 1)
    ia, ib = np.triu_indices(V, 1)
    return np.concatenate([t1.ravel(), t2[io, jo][:, ia, ib].ravel(), np.asarray(extra, dtype=complex)])


@pytest.mark.parametrize("O,V,seed", WIDE)
@pytest.mark.parametrize("fold", [True, False])
def test_residual_step_wide_virtual_space(dev, O, V, seed, fold):
    """Residual step (reference form) with several epilogue tiles, with the
    F_vv terms folded into the ring block and as a separate product."""
    F, A, eps, ints = _system(O, V, seed, dev)
    t1, t2 = rand_amplitudes(O, V, seed + 1)
    E = 0.021 + 0.004j
    solver = SOCI(ints, _dev(F, dev), eps, singles=True, fold_fvv=fold)
    assert (solver.ring_f is not None) == fold
    t = _dev(np.concatenate([t1.ravel(), t2.ravel()]), dev)
    tn, r = solver.new_vector(), solver.new_vector()
    solver.step(t, tn, r, energy=torch.tensor([E], dtype=torch.complex128, device=dev))
    r1, r2 = so.cisd_so_residual(F, A / 2, t1, t2, E, O)
    D1, D2 = so.denominators(eps[:O], eps[O:])
    g1, g2 = (x.cpu().numpy() for x in solver.split(r))
    n1, n2 = (x.cpu().numpy() for x in solver.split(tn))
    scale = max(1.0, np.abs(r2).max())
    assert np.abs(g1 - r1).max() < 1e-13 * scale and np.abs(g2 - r2).max() < 1e-13 * scale
    assert np.abs(n1 - (t1 + r1 / D1)).max() < 1e-12 and np.abs(n2 - (t2 + r2 / D2)).max() < 1e-12


@pytest.mark.parametrize("O,V,seed", WIDE)
def test_residual_step_in_place_update(dev, O, V, seed):
    """t_new may alias t (the header allows it): the same update as into a
    separate vector."""
    F, A, eps, ints = _system(O, V, seed, dev)
    t1, t2 = rand_amplitudes(O, V, seed + 5)
    solver = SOCI(ints, _dev(F, dev), eps, singles=True)
    Ed = torch.tensor([0.01 - 0.003j], dtype=torch.complex128, device=dev)
    t = _dev(np.concatenate([t1.ravel(), t2.ravel()]), dev)
    t_sep, r1, r2 = solver.new_vector(), solver.new_vector(), solver.new_vector()
    solver.step(t, t_sep, r1, energy=Ed)
    solver.step(t, t, r2, energy=Ed)
    assert torch.equal(t, t_sep) and torch.equal(r1, r2)


@pytest.mark.parametrize("O,V,seed", WIDE + [(6, 8, 5)])
@pytest.mark.parametrize("singles", [True, False])
def test_packed_sigma_matches_dense_and_oracle(dev, O, V, seed, singles):
    """sigma mode on packed vectors [t1 | t2 over (i<j, a<b)] (the Davidson
    layout) equals the packed image of the dense sigma and the oracle's
    Hermitian CISD matrix product (singles) or the reference's CID doubles
    sigma; the packed energy equals the dense one."""
    F, A, eps, ints = _system(O, V, seed, dev)
    t1, t2 = rand_amplitudes(O, V, seed + 2)
    if not singles:
        t1 = np.zeros_like(t1)
    c0 = 0.9 + 0.15j
    solver = SOCI(ints, _dev(F, dev), eps, singles=singles, fov_coupling=singles)
    dense_in = _dev(np.concatenate([t1.ravel(), t2.ravel()]), dev)
    dense_out = solver.new_vector()
    solver.sigma(dense_in, dense_out, c0=c0)
    p_in = _dev(_packed(t1, t2, O, V), dev)
    p_out = torch.zeros_like(p_in)
    solver.sigma(p_in, p_out, c0=c0, packed=True)
    d1, d2 = (x.cpu().numpy() for x in solver.split(dense_out))
    want_p = _packed(d1, d2, O, V)
    assert np.array_equal(p_out.cpu().numpy()[:O * V], want_p[:O * V]) or not singles
    scale = max(1.0, np.abs(want_p).max())
    assert np.abs(p_out.cpu().numpy() - want_p).max() < 1e-14 * scale
    W = so.blocks_from_eri(A / 2, O)
    if singles:
        from oracle import davidson
        s0, s1, s2 = davidson.sigma(F, W, c0, t1, t2, O)
    else:
        s1 = np.zeros_like(t1)
        s2 = so.cid_so_residual(F, A / 2, t2, 0.0, O) + (c0 - 1.0) * W['vvoo'].transpose(2, 3, 0, 1)
    assert np.abs(p_out.cpu().numpy() - _packed(s1, s2, O, V)).max() < 1e-13 * scale
    e_dense = complex(solver.energy(dense_in, out=torch.zeros(1, dtype=torch.complex128, device=dev)).cpu()[0])
    e_pack = complex(solver.energy(p_in, out=torch.zeros(1, dtype=torch.complex128, device=dev), packed=True)
                     .cpu()[0])
    assert abs(e_dense - e_pack) < 1e-14 * max(1.0, abs(e_dense))


@pytest.mark.parametrize("O,V,seed", WIDE + [(6, 8, 5)])
@pytest.mark.parametrize("fold", [True, False])
def test_gauss3m_sigma_and_residual_match_oracle(dev, O, V, seed, fold):
    """SOCI(gauss3m=True), the PPL and ring products in the three-product
    complex form: the packed Hermitian sigma against the oracle's CISD
    matrix product and the dense residual step against the reference's
    residual, at the bounds the four-product form meets."""
    F, A, eps, ints = _system(O, V, seed, dev)
    t1, t2 = rand_amplitudes(O, V, seed + 4)
    c0 = 0.8 - 0.2j
    herm = SOCI(ints, _dev(F, dev), eps, singles=True, fov_coupling=True, fold_fvv=fold, gauss3m=True)
    p_in = _dev(_packed(t1, t2, O, V), dev)
    p_out = torch.zeros_like(p_in)
    herm.sigma(p_in, p_out, c0=c0, packed=True)
    W = so.blocks_from_eri(A / 2, O)
    from oracle import davidson
    _, s1, s2 = davidson.sigma(F, W, c0, t1, t2, O)
    want = _packed(s1, s2, O, V)
    scale = max(1.0, np.abs(want).max())
    assert np.abs(p_out.cpu().numpy() - want).max() < 1e-13 * scale
    solver = SOCI(ints, _dev(F, dev), eps, singles=True, fold_fvv=fold, gauss3m=True)
    E = -0.21 + 0.003j
    t = _dev(np.concatenate([t1.ravel(), t2.ravel()]), dev)
    tn, r = solver.new_vector(), solver.new_vector()
    solver.step(t, tn, r, energy=torch.tensor([E], dtype=torch.complex128, device=dev))
    g1, g2 = (x.cpu().numpy() for x in solver.split(r))
    r1, r2 = so.cisd_so_residual(F, A / 2, t1, t2, E, O)
    scale = max(1.0, np.abs(r1).max(), np.abs(r2).max())
    assert np.abs(g1 - r1).max() < 1e-13 * scale
    assert np.abs(g2 - r2).max() < 1e-13 * scale
