"""The attention operators under autograd (CPU, with a stand-in for the device kernel): what they write
counts as written, they record no derivative, and transforms that take one are refused."""

import pytest
import torch
import torch.autograd.forward_ad as forward_ad

import hilberta_amd  # noqa: F401  (registers the ops)

OPS = torch.ops.hilberta_hip


def _paired(q, out, lse=None):
    table = torch.zeros(1, 1, dtype=torch.int32)
    return OPS.paired_fwd(q, q, q, out, lse, table, table, table[0], 0, 64, 1.0, True, 0)


def _sparse(q, out, lse=None):
    table = torch.zeros(1, 1, dtype=torch.int32)
    return OPS.sparse_fwd(q, q, q, out, lse, table, table[0], 0, 1.0, True, 0)


@pytest.fixture(params=[_paired, _sparse])
def attend(request):
    def kernel(q, k, v, out, lse, *rest):
        out.fill_(2.0)
        if lse is not None:
            lse.fill_(3.0)

    with torch.library._scoped_library("hilberta_hip", "IMPL") as lib:
        lib.impl("paired_fwd", kernel, "CPU")
        lib.impl("sparse_fwd", kernel, "CPU")
        yield request.param


def test_written_arguments_count(attend):
    q, out, lse = torch.ones(4), torch.zeros(4), torch.zeros(4)
    attend(q, out, lse)
    assert (out._version, lse._version, q._version) == (1, 1, 0)
    attend(q, out)
    assert (out._version, lse._version) == (2, 1)
    with torch.inference_mode():
        attend(q, out)
        made_there = torch.zeros(4)
        attend(q, made_there)
    assert out._version == 3
    attend(q, made_there)   # (an inference tensor has no version)
    assert (out == 2).all() and (lse == 3).all() and (made_there == 2).all()


def test_overwriting_a_saved_tensor_fails_its_backward(attend):
    w, out = torch.ones(4, requires_grad=True), torch.zeros(4)
    y = (out * w).sum()
    attend(torch.ones(4), out)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()


def test_no_derivative(attend):
    q, out = torch.ones(4, requires_grad=True), torch.zeros(4)
    attend(q, out)
    assert not out.requires_grad and out._version == 1
    leaf = torch.zeros(4, requires_grad=True)
    attend(torch.ones(4), leaf)
    assert leaf.is_leaf and leaf._version == 1

    def total(q):
        out = torch.zeros(4)
        attend(q, out)
        return out.sum()

    with pytest.raises(RuntimeError, match="torch.func"):
        torch.func.grad(total)(torch.ones(4))
    with forward_ad.dual_level(), pytest.raises(NotImplementedError, match="forward AD"):
        attend(forward_ad.make_dual(torch.ones(4), torch.ones(4)), out)
