"""The wait for the device in front of a call: torch's own function where it has
one and the device is in use, torch.cuda.synchronize otherwise (host-only)."""
import pytest
import torch

from lap_amd import solver as S


@pytest.mark.parametrize("present,initialised,want", [(True, True, "short"), (True, False, "public"),
                                                      (False, True, "public"),
                                                      (False, False, "public")])
def test_which_wait(monkeypatch, present, initialised, want):
    calls = []
    monkeypatch.setattr(S, "_device_sync", (lambda: calls.append("short")) if present else None)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: initialised)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: calls.append("public"))
    S._sync()
    assert calls == [want]
