"""The unrolled iterations call the projections of their system matrix also
where a caller wraps them on the object or on the class."""
from pytomography_amd import _lib
from pytomography_amd.projectors.SPECT import SPECTSystemMatrix
from pytomography_amd.unrolled import UnrolledBSREM


class _Fused(SPECTSystemMatrix):
    fused = True

    def __init__(self):
        pass

    def _project(self, x, k, entry, planes=False):
        return "projected"

    def _backward(self, p, k, mode, planes=False):
        return "back projected"


def _unrolled():
    u = UnrolledBSREM.__new__(UnrolledBSREM)
    u.sm = _Fused()
    return u


def test_wrapper_on_the_object():
    u = _unrolled()
    u.sm.forward = lambda x, k: ("object", k)
    u.sm.backward_adjoint = lambda p, k: ("adjoint", k)
    assert u._forward(None, 3) == ("object", 3)
    assert u._backward(None, 3, _lib.BP_ADJOINT) == ("adjoint", 3)
    assert u._backward(None, 3) == "back projected"


def test_wrapper_on_the_class(monkeypatch):
    monkeypatch.setattr(SPECTSystemMatrix, "backward", lambda self, p, k=None: ("class", k))
    u = _unrolled()
    assert u._backward(None, 3) == ("class", 3)
    assert u._forward(None, 3) == "projected"
