"""Real-node evaluation of complex directions (CPU): the interpolation weights.

polytensors_amd/_complex.py recovers a complex-direction coefficient P_k(i) from
real evaluations P_k(lam_m), P_k a real polynomial of degree <= k <= K. These
tests check the weights against the defining identity on monomials and on a
random polynomial (the GPU round trip through the plane kernels is in
tests/test_gpu_complex.py).
"""

import pytest
import torch

from polytensors_amd import PolyTensor, _complex, _fused_activation, _fused_attention


def test_weights_evaluate_every_monomial_at_i():
    for degree in range(0, 9):
        nodes, weights = _complex.nodes_and_weights(degree)
        assert len(set(nodes)) == degree + 1 and all(isinstance(x, float) for x in nodes)
        for j in range(degree + 1):
            got = sum(w * lam ** j for w, lam in zip(weights, nodes))
            assert abs(got - 1j ** j) < 1e-9 * max(1.0, max(abs(x) for x in nodes) ** j)


def test_weights_on_a_random_polynomial():
    g = torch.Generator().manual_seed(0)
    for degree in (1, 3, 5):
        coeffs = torch.randn(degree + 1, generator=g, dtype=torch.float64).tolist()
        nodes, weights = _complex.nodes_and_weights(degree)
        p = lambda z: sum(c * z ** j for j, c in enumerate(coeffs))  # noqa: E731
        assert abs(sum(w * p(x) for w, x in zip(weights, nodes)) - p(1j)) < 1e-12 * sum(abs(c) for c in coeffs) * 2 ** degree


def _direction(shape, degree, dtype, complex_=True):
    """A series of the given shape without its memory (one element, expanded)."""
    wide = {torch.float32: torch.complex64, torch.float64: torch.complex128}[dtype] if complex_ else dtype
    return PolyTensor((torch.zeros(1, dtype=dtype).expand(shape),) + (torch.zeros(1, dtype=wide).expand(shape),) * degree)


# Both sides of the rule that runs the interpolation nodes of an attention as one batch.
@pytest.mark.parametrize("heads,L,S,d,degree,dtype,one_launch", [
    (24, 512, 512, 64, 3, torch.float32, True), (8, 1024, 1024, 128, 3, torch.float32, True),
    (64, 1024, 1024, 128, 2, torch.float32, False), (24, 1024, 1024, 128, 1, torch.float32, True),
    (64, 512, 512, 64, 2, torch.float32, False), (64, 1024, 1024, 32, 2, torch.float32, True), (1800, 64, 64, 32, 2, torch.float32, False), (256, 256, 256, 128, 1, torch.float32, False),
    (64, 4, 1000, 128, 1, torch.float32, False), (1, 64, 64, 128, 2, torch.float32, True),
    (1024, 16, 16, 32, 1, torch.float32, True), (2048, 16, 16, 32, 1, torch.float32, False),
    (1, 1024, 1024, 128, 3, torch.float64, False), (8, 1024, 1024, 32, 3, torch.float64, True),
    (24, 512, 512, 128, 1, torch.float64, False), (1, 16, 16, 16, 9, torch.float64, False), (0, 16, 16, 16, 1, torch.float64, False)])
def test_attention_nodes_in_one_launch(heads, L, S, d, degree, dtype, one_launch):
    q, k, v = (_direction((heads, n, d), degree, dtype) for n in (L, S, S))
    assert _fused_attention._stacks_nodes(q, k, v, None, False, degree) is one_launch
    assert not _fused_attention._stacks_nodes(q, k, v, torch.zeros(2, L, S, dtype=torch.bool), False, degree)


def test_attention_nodes_in_one_launch_by_kernel():
    """Shapes that are no longer launch-bound: an ordinary operand or an additive mask takes the other kernel."""
    q, k, v = (_direction((24, 512, 64), 3, torch.float32) for _ in range(3))
    stacks = _fused_attention._stacks_nodes
    assert stacks(q, k, v, torch.ones(512, 512, dtype=torch.bool), False, 3)
    q, k, v = (_direction((8, 512, 64), 3, torch.float32) for _ in range(3))   # 64 workgroups
    assert stacks(q, k, v, None, False, 3)
    assert not stacks(q, torch.zeros(8, 512, 64), v, None, False, 3)
    assert not stacks(q, k, v, torch.zeros(512, 512), False, 3)
    q, k, v = (_direction((64, 1024, 64), 3, torch.float32) for _ in range(3))   # 1024 workgroups
    assert stacks(q, k, v, None, True, 3) and not stacks(q, k, v, None, False, 3)


# Causal calls of the kernel that shares few workgroups' keys out over the chip: the batch's own workgroups count too.
@pytest.mark.parametrize("heads,T,d,degree,one_launch", [
    (16, 361, 64, 2, True), (8, 361, 64, 2, False), (8, 512, 64, 1, False), (16, 512, 64, 1, True),
    (48, 512, 64, 2, True), (64, 512, 64, 2, False), (1, 1024, 128, 3, False)])
def test_causal_attention_nodes_in_one_launch(heads, T, d, degree, one_launch):
    q, k, v = (_direction((heads, T, d), degree, torch.float64) for _ in range(3))
    assert _fused_attention._stacks_nodes(q, k, v, None, True, degree) is one_launch
    # a mask beside the causal rule becomes one mask: the rule of masked calls
    keep = torch.ones(T, T, dtype=torch.bool)
    assert (_fused_attention._stacks_nodes(q, k, v, keep, True, degree)
            is _fused_attention._stacks_nodes(q, k, v, keep, False, degree))


@pytest.mark.parametrize("degree,numel,dtype,one_pass", [
    (1, 1 << 21, torch.float64, True), (1, (1 << 21) + 1, torch.float64, False), (2, 1 << 24, torch.float64, True),
    (1, 1 << 24, torch.float32, True), (9, 4, torch.float32, False)])
def test_activation_in_one_pass(degree, numel, dtype, one_pass):
    assert _fused_activation._one_pass(_direction((numel,), degree, dtype)) is one_pass
