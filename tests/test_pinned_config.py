"""SDPV_GEMM_CONFIG pins the tile configuration of every product that is large enough to be tuned, short inner
dimensions included."""
import types

import pytest

from sdpvibe_amd import rns


@pytest.mark.parametrize("kc", [1, 32, 33, 70, 96, 97, 600])
@pytest.mark.parametrize("forced", [None, *rns.GEMM_CONFIGS])
def test_pinned_configuration_is_taken(monkeypatch, kc, forced):
    monkeypatch.setattr(rns, "FORCED", forced)
    monkeypatch.setattr(rns, "_measure", lambda *a: -7)           # what tuning would pick
    R = types.SimpleNamespace(L=24, KPAD=rns.RNS.KPAD)
    R.kp = lambda k: rns.RNS.kp(R, k)
    kp = rns.RNS.kp_product(R, kc)
    assert kp >= kc and kp % (64 if kc > 96 else 32) == 0 and kp - kc < 64
    monkeypatch.setattr(rns, "_tuned", {})
    assert rns.tuned_config(R, 1, 2048, 2048, kp) == (-7 if forced is None else forced)
