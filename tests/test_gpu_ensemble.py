"""Ensemble member synthesis in one batch (needs an MI355X).

``ensemble_grid_fields`` / ``EnsembleSynthesis`` replace the reference's
member loop in ``grid_fields`` (da/ensemble.py:547-579): every member's u, v,
theta, qv, ln ps and the potentials psi = inverse(inverse_laplacian(zeta)),
chi = the same of D, from one grouped batch.  Checked against the FP64 oracle
per member, bit for bit against the single operations the reference calls
(the inverse Laplacian fused into the pack is the spectral operator's own
arithmetic), and across graph replays.
"""
from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest

from oracle.sht import OracleTransform, red_spectrum

from _helpers import hip_transform, rel_err

pytestmark = pytest.mark.gpu

TOL = {"float32": 1e-6, "bf16x6": 1e-6}


@pytest.fixture(scope="module")
def oracle():
    return OracleTransform.create(63, dealias_factor=1.0)


def _members(o, R, L, seed=0):
    T = o.grid.truncation
    out = []
    for k in range(R):
        s = seed + 100 * k
        out.append({
            "vorticity": o.project(red_spectrum(T, (L,), seed=s + 1, scale=1e-5)),
            "divergence": o.project(red_spectrum(T, (L,), seed=s + 2, scale=2e-6)),
            "theta": o.project(red_spectrum(T, (L,), seed=s + 3, scale=10.0, mean=300.0)),
            "qv": o.project(red_spectrum(T, (L,), seed=s + 4, scale=1e-3, mean=5e-3)),
            "log_surface_pressure": o.project(red_spectrum(T, (), seed=s + 5, scale=1e-2,
                                                           mean=11.5)),
        })
    return out


def _np(t):
    return t.detach().cpu().numpy()


@pytest.mark.parametrize("precision", ["float32", "bf16x6"])
def test_every_member_matches_the_oracle_and_the_single_operations(oracle, precision):
    import torch
    from arwen_spectral import VorticityDivergenceOperator, ensemble_grid_fields

    o = oracle
    tr = hip_transform(o, precision)
    R, L = 4, 3
    host = _members(o, R, L)
    dev = torch.device("cuda", torch.cuda.current_device())
    c64 = lambda a: torch.from_numpy(np.ascontiguousarray(a).astype(np.complex64)).to(dev)
    members = [{k: c64(v) for k, v in m.items()} for m in host]
    got = ensemble_grid_fields(tr, members)
    assert set(got) == {"u", "v", "theta", "qv", "lnps", "psi", "chi"}
    assert tuple(got["u"].shape) == (R, L, *tr.grid.shape)
    assert tuple(got["lnps"].shape) == (R, *tr.grid.shape)
    op = VorticityDivergenceOperator(tr)
    for k in range(R):
        h = {n: _np(members[k][n]).astype(np.complex128) for n in members[k]}
        u, v = o.wind_from_vordiv(h["vorticity"], h["divergence"])
        want = {"u": u, "v": v, "theta": o.inverse(h["theta"]), "qv": o.inverse(h["qv"]),
                "lnps": o.inverse(h["log_surface_pressure"]),
                "psi": o.inverse(o.inverse_laplacian(h["vorticity"])),
                "chi": o.inverse(o.inverse_laplacian(h["divergence"]))}
        for n, w in want.items():
            err = rel_err(got[n][k], w)
            assert err <= TOL[precision], (k, n, err)
        # the reference's own calls, one member at a time
        su, sv = op.wind_from_vordiv(members[k]["vorticity"], members[k]["divergence"])
        single = {"u": su, "v": sv, "theta": tr.inverse(members[k]["theta"]),
                  "lnps": tr.inverse(members[k]["log_surface_pressure"]),
                  "psi": tr.inverse(tr.inverse_laplacian(members[k]["vorticity"])),
                  "chi": tr.inverse(tr.inverse_laplacian(members[k]["divergence"]))}
        for n, t in single.items():
            assert np.array_equal(_np(got[n][k]), _np(t)), (k, n)


def test_state_objects_graph_replays_and_refusals(oracle):
    import torch
    from arwen_spectral import EnsembleSynthesis

    o = oracle
    tr = hip_transform(o, "bf16x6")
    R, L = 3, 2
    dev = torch.device("cuda", torch.cuda.current_device())
    host = _members(o, R, L, seed=7)
    states = [SimpleNamespace(atmosphere=SimpleNamespace(
        **{k: torch.from_numpy(v.astype(np.complex64)).to(dev) for k, v in m.items()}))
        for m in host]
    ens = EnsembleSynthesis(tr, R, L, names=("psi", "theta", "lnps"))
    assert set(ens.inputs) == {"vorticity", "theta", "log_surface_pressure"}
    ens.load(states)
    eager = {n: t.clone() for n, t in ens.run().items()}
    torch.cuda.synchronize()
    for _ in range(3):
        out = ens.run(graph=True)
        torch.cuda.synchronize()
        for n in eager:
            assert np.array_equal(_np(out[n]), _np(eager[n])), n
        ens.run()  # eager work between the replays
        torch.cuda.synchronize()
    for k in range(R):
        err = rel_err(eager["psi"][k], o.inverse(o.inverse_laplacian(
            host[k]["vorticity"].astype(np.complex64).astype(np.complex128))))
        assert err <= 1e-6
    with pytest.raises(ValueError, match="expected 3 members"):
        ens.load(states[:2])
    with pytest.raises(ValueError, match="unknown grid fields"):
        EnsembleSynthesis(tr, R, L, names=("w",))


def test_load_holds_few_copies_of_host_members():
    """Host members pass through the device a few fields at a time: no more
    than the fields that wait together and the one being converted (complex128
    first, so three times its bytes) are live beside the inputs."""
    import torch

    from arwen_spectral import EnsembleSynthesis
    from arwen_spectral.ensemble import _HELD_BYTES, _TOGETHER_BYTES

    o = OracleTransform.create(63, dealias_factor=1.0)
    tr = hip_transform(o, "float32")
    rng = np.random.default_rng(0)
    for R, L in ((30, 60), (4, 300)):  # fields of 1.9 MiB and, one by one, 9.4 MiB
        ens = EnsembleSynthesis(tr, R, L, ("theta", "qv"))
        x = rng.standard_normal((L, 64, 64)) + 1j * rng.standard_normal((L, 64, 64))
        members = [{"theta": x + k, "qv": x - k} for k in range(R)]
        field = L * 64 * 64 * 8
        assert 2 * R * field > 2 * (_HELD_BYTES + 4 * field) or field > _TOGETHER_BYTES
        ens.load(members)  # the caching allocator's blocks exist
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        ens.load(members)
        waiting = _HELD_BYTES + field if field <= _TOGETHER_BYTES else field
        assert torch.cuda.max_memory_allocated() - before <= waiting + 3 * field + (4 << 20)
        for k in (0, R // 2, R - 1):
            for name, sign in (("theta", 1), ("qv", -1)):
                assert np.array_equal(_np(ens.inputs[name][k]),
                                      (x + sign * k).astype(np.complex64))


def test_load_from_the_inputs_themselves_keeps_the_members_order():
    """Members given as views of the stacked inputs are copied one after the
    other: a shift by one member, and a later member that reads an earlier one."""
    import torch

    from arwen_spectral import EnsembleSynthesis

    o = OracleTransform.create(31, dealias_factor=1.0)
    tr = hip_transform(o, "float32")
    R, L = 6, 40
    ens = EnsembleSynthesis(tr, R, L, ("theta", "lnps"))
    gen = torch.Generator(device="cuda").manual_seed(3)

    def fresh(like):
        return torch.view_as_complex(torch.randn((*like.shape, 2), generator=gen, device="cuda"))

    names = {"theta": "theta", "log_surface_pressure": "log_surface_pressure"}
    for trial in range(3):
        for t in ens.inputs.values():
            t.copy_(fresh(t))
        new = {s: fresh(ens.inputs[s][0]) for s in names}
        for source in (lambda t, k: t[k + 1] if k + 1 < R else None,       # forward shift
                       lambda t, k: t[R - 1 - k],                          # reversal in place
                       lambda t, k: t[0].mT if k else None):               # a strided view
            want = {s: ens.inputs[s].clone() for s in names}
            for s in names:
                for k in range(R):  # one after the other
                    src = source(want[s], k)
                    want[s][k].copy_(new[s] if src is None else src)
            members = []
            for k in range(R):
                members.append({s: new[s] if source(ens.inputs[s], k) is None
                                else source(ens.inputs[s], k) for s in names})
            ens.load(members)
            for s in names:
                assert torch.equal(ens.inputs[s], want[s])


@pytest.mark.parametrize("L,calls", [(40, 1), (300, 0)])  # fields of 1.3 and 9.4 MiB
def test_the_largest_field_decides_how_members_are_copied(monkeypatch, L, calls):
    """Small members go in one joint copy; beside large fields the small ones
    are copied one by one as well."""
    import torch

    from arwen_spectral import EnsembleSynthesis

    o = OracleTransform.create(63, dealias_factor=1.0)
    ens = EnsembleSynthesis(hip_transform(o, "float32"), 2, L, ("theta", "lnps"))
    gen = torch.Generator(device="cuda").manual_seed(5)
    members = [{s: torch.randn(buf.shape[1:], generator=gen, dtype=buf.dtype, device="cuda")
                for s, buf in ens.inputs.items()} for _ in range(2)]
    joint, copy = [], torch._foreach_copy_
    monkeypatch.setattr(torch, "_foreach_copy_", lambda a, b: (joint.append(len(a)), copy(a, b)))
    ens.load(members)
    assert len(joint) == calls
    for k, member in enumerate(members):
        for s, buf in ens.inputs.items():
            assert torch.equal(buf[k], member[s])
