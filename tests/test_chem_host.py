"""Host-side chemistry of the library (no GPU): boundary states and the
parser of the 9-species test mechanism, against the CPU oracle; the
production rates Jex forms beside the Jacobian, against Fex; tables with more
transport entries than species, and with indices of no species."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O
from oracle.chem_inp import read_cheminp
from shared_cfd_amd import chem

from chem_cases import NO27, no27_plus_h2o2, repeated_trans


@pytest.fixture(scope="module")
def mechs(tmp_path_factory):
    d = tmp_path_factory.mktemp("m")
    c, t = chem.write_synthetic_mechanism(3, str(d / "syn"))
    p9 = no27_plus_h2o2(str(d / "no27"))
    return {"syn": (chem.parse(c, t), read_cheminp(c, chem.MW_INP, t)),
            "no27_9": (chem.parse(p9), read_cheminp(p9, chem.MW_INP))}


@pytest.mark.parametrize("which", ["syn", "no27_9"])
def test_boundary_state_matches_oracle_bitwise(mechs, which):
    lm, om = mechs[which]
    assert lm.ns == 9
    rng = np.random.default_rng(0)
    for T in (300.0, 1000.0, 1500.0, 2400.0):
        rel = rng.random(9) + 0.01
        w, vhi, dhi = chem.boundary_state(lm, 1.01325e5, T, rel)
        vrho, rho, E = O.chem_rho_rel2abs(om, 1.01325e5, T, rel)
        T1, out, it = O.chem_calc_t(om, vrho, rho, E, T)
        ns = 9
        assert w[0] == rho and w[3] == 1.01325e5
        assert np.array_equal(w[4:4 + ns], vrho / rho)
        assert w[ns + 4] == out[0]                        # gamma
        assert w[ns + 5] == E + 1.01325e5 / rho           # H (u = v = 0)
        assert w[ns + 6] == 8.3144621e3 / out[1]          # R
        assert w[ns + 7] == out[2]                        # mu
        assert np.array_equal(vhi, out[3 + ns:3 + 2 * ns]) and np.array_equal(dhi, out[3:3 + ns])


def test_no27_with_h2o2_parses(mechs):
    lm, om = mechs["no27_9"]
    assert (lm.ns, lm.nr) == (9, 9)
    a, b = chem.Mech.from_buffer_copy(bytes(lm)), om
    a.rtol = a.atol = b.rtol = b.atol = 0.0
    assert bytes(a) == bytes(b)


@pytest.mark.parametrize("which", ["syn", "no27_9"])
def test_jex_production_rates_are_fex_bit_for_bit(mechs, which):
    """Jex (FJ.f90:454-708) accumulates dn/dt with the same rates, in the same
    order, as Fex (:152-300); the point-implicit update takes f from it
    instead of a second evaluation of every rate, which is exact only if the
    two agree in every bit.  States: ignition-like mixtures at 300-3000 K (both
    NASA ranges), with some species near the 1e-30 floor."""
    lm, _ = mechs[which]
    so = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host", "libchem_host.so")
    L = ctypes.CDLL(so)
    dp = ctypes.POINTER(ctypes.c_double)
    L.host_fex_jex.argtypes = [ctypes.c_void_p, ctypes.c_int, dp, dp, dp]
    rng = np.random.default_rng(7)
    ns, n = lm.ns, 4000
    conc = 10.0 ** rng.uniform(-12, -5, (n, ns))
    conc[rng.random((n, ns)) < 0.1] = 1e-30
    T = rng.uniform(300.0, 3000.0, (n, 1))
    x = np.ascontiguousarray(np.hstack([conc, T]))
    f, g = np.zeros_like(x), np.zeros_like(x)
    assert L.host_fex_jex(ctypes.addressof(lm), n, x.ctypes.data_as(dp), f.ctypes.data_as(dp),
                          g.ctypes.data_as(dp)) == 0
    assert np.all(np.isfinite(f)) and np.max(np.abs(f[:, :ns])) > 0
    assert np.array_equal(f, g)


@pytest.mark.parametrize("extra", [0, 1, 2, 5])
def test_more_transport_entries_than_species(tmp_path, extra):
    """A trans.inp that lists species twice gives up to 16 entries for any
    species count: every index stays in its array, and the viscosity is the
    oracle's, bit for bit."""
    t = repeated_trans(str(tmp_path), extra)
    lm, om = chem.parse(NO27, t), read_cheminp(NO27, chem.MW_INP, t)
    assert (lm.ns, lm.nt) == (om.ns, om.nt) == (8, 7 + extra)
    table = tmp_path / "mech.bin"
    table.write_bytes(bytes(lm))
    rel = np.random.default_rng(extra).random(8) + 0.01
    exe = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host", "chem_bounds")
    r = subprocess.run([exe, str(table), "1500.0", *[repr(float(v)) for v in rel]], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    vrho, rho, E = O.chem_rho_rel2abs(om, 1.01325e5, 1500.0, rel)
    mu = O.chem_calc_t(om, vrho, rho, E, 1500.0)[1][2]
    assert float(r.stdout) == mu
    assert chem.boundary_state(lm, 1.01325e5, 1500.0, rel)[0][8 + 7] == mu


TRANSPORT = [("tr2th[0]", 9), ("tr2th[1]", -1), ("nt", 17)]
REACTIONS = [("num_nu[0][0]", 4), ("ind_nu[1][1][0]", 9), ("ind_nu[0][0][0]", -1), ("num_m[4]", 17), ("ind_m[4][0]", 9)]


@pytest.mark.parametrize("entry,value", TRANSPORT + REACTIONS)
def test_tables_with_indices_of_no_species_are_refused(mechs, entry, value):
    """shcfd_chem_eval looks at the table before it looks for a GPU; the
    boundary states use its transport entries alone."""
    m = chem.Mech.from_buffer_copy(bytes(mechs["syn"][0]))
    assert m.nt > 1 and m.exist_m[4] == 1 and m.num_m[4] > 0
    name, *idx = entry.replace("]", "").split("[")
    if idx:
        a = getattr(m, name)
        for i in idx[:-1]:
            a = a[int(i)]
        a[int(idx[-1])] = value
    else:
        setattr(m, name, value)
    x, out, st = np.zeros(10), np.zeros(10), np.zeros(1, np.int32)
    dp, ip = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int)
    L = chem._lib()
    for call in (L.shcfd_chem_eval, L.shcfd_chem_eval_noalloc):
        rc = call(ctypes.byref(m), chem.FEX, 1, x.ctypes.data_as(dp), out.ctypes.data_as(dp), st.ctypes.data_as(ip),
                  ctypes.c_double(0.0))
        assert rc == 1  # SHCFD_E_ARG
    if (entry, value) in TRANSPORT:
        with pytest.raises(ValueError):
            chem.boundary_state(m, 1.01325e5, 1000.0, np.ones(9))
    else:
        chem.boundary_state(m, 1.01325e5, 1000.0, np.ones(9))
