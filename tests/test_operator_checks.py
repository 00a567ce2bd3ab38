"""CPU checks of the operator layer: host memory that a kernel would follow is
refused, and replaced module-level operators are called.  Tensors that only claim to be on the GPU reach the checks; nothing is launched."""
import pytest
import torch

from localmoe35ba3b_amd import _lib, router
from localmoe35ba3b_amd.operators import int8, w8a8


class OnGpu(torch.Tensor):
    is_cuda = True


def gpu(t):
    return t.as_subclass(OnGpu)


@pytest.fixture
def launches(monkeypatch):
    names = []
    monkeypatch.setattr(_lib, 'call', lambda name, *args: names.append(name))
    monkeypatch.setattr(_lib, 'stream', lambda device=None: 0)
    return names


X = torch.zeros(1, 256, dtype=torch.bfloat16)
TABLE = torch.zeros(4, 5, dtype=torch.int64)
OPERATORS = {
    'w8a16': lambda t: int8.grouped_linear(gpu(X), t, 4, 64, 0, True),
    'w8a8': lambda t: w8a8.grouped_linear(gpu(X), t, 4, 64, 0, True),
    'w8a8 quantized': lambda t: w8a8.grouped_gemv(gpu(X.to(torch.int8)), gpu(torch.zeros(1, 2)), t,
                                                  4, 64, 0, True),
    'combine': lambda t: int8.ordered_reduce(gpu(torch.zeros(4, 64, dtype=torch.bfloat16)), t,
                                             gpu(torch.zeros(1, 4))),
}


@pytest.mark.parametrize('operator', OPERATORS)
def test_descriptor_table_must_be_on_the_gpu(launches, operator):
    run = OPERATORS[operator]
    for table in (TABLE, gpu(TABLE.int()), gpu(TABLE[:3])):
        with pytest.raises(ValueError, match='descriptor table'):
            run(table)
    assert launches == []
    run(gpu(TABLE))
    assert len(launches) == 1


def _experts():
    bank = [gpu(torch.zeros(s, dtype=d)) for s, d in (
        ((6, 256, 256), torch.int8), ((6, 256, 2), torch.float32),
        ((6, 256, 128), torch.int8), ((6, 256, 1), torch.float32))]
    return int8.Int8Experts(0, {'q': bank[0], 'scale': bank[1]}, {'q': bank[2], 'scale': bank[3]})


@pytest.mark.parametrize('swap', [False, True])
def test_experts_refuse_host_routing(launches, monkeypatch, swap):
    if swap:
        monkeypatch.setattr(int8, 'grouped_linear', w8a8.grouped_linear)
    experts, ids, weights = _experts(), torch.zeros(1, 4, dtype=torch.int64), torch.zeros(1, 4)
    for i, w in ((ids, gpu(weights)), (gpu(ids), weights), (gpu(ids), gpu(weights[:, :3]))):
        with pytest.raises(ValueError, match='CUDA'):
            experts(gpu(X), i, w)
    if not swap:
        assert launches == []
        experts(gpu(X), gpu(ids), gpu(weights))
        assert launches == ['lm_w8a16_experts_decode']


@pytest.mark.parametrize('name', ['build_descriptors', 'grouped_linear', 'swiglu',
                                  'ordered_reduce'])
def test_experts_call_replaced_operators(launches, monkeypatch, name):
    """One decode token runs a program's own operator where it replaced one at
    module level, and the fused launches where it did not."""
    empty = torch.empty
    monkeypatch.setattr(torch, 'empty', lambda *a, device=None, **kw: gpu(empty(*a, **kw)))
    experts, ids = _experts(), gpu(torch.zeros(1, 4, dtype=torch.int64))
    experts(gpu(X), ids, gpu(torch.zeros(1, 4)))
    assert launches == ['lm_w8a16_experts_decode']
    calls, original = [], getattr(int8, name)
    monkeypatch.setattr(int8, name, lambda *a, **kw: calls.append(name) or original(*a, **kw))
    experts(gpu(X), ids, gpu(torch.zeros(1, 4)))
    assert calls == [name] * (2 if name == 'grouped_linear' else 1)
    assert launches[1:] == ['lm_expert_table', 'lm_w8a16_grouped_gemv', 'lm_swiglu',
                            'lm_w8a16_grouped_gemv', 'lm_ordered_reduce']


def test_router_without_memory_for_its_workspace(launches, monkeypatch):
    """A router call that finds no memory for its scratch runs the form without."""
    new_empty, args = torch.Tensor.new_empty, []

    def full(self, size, dtype=None, **kw):
        if dtype is torch.uint8:
            raise torch.OutOfMemoryError('no memory')
        return new_empty(self, size, dtype=dtype or self.dtype, **kw)

    monkeypatch.setattr(OnGpu, 'new_empty', full)
    monkeypatch.setattr(_lib, 'call', lambda name, *a: args.append((name, a[-3:-1])))
    router.router_topk(gpu(torch.zeros(2048, 2048, dtype=torch.bfloat16)),
                       gpu(torch.zeros(256, 2048, dtype=torch.bfloat16)), 8)
    assert args == [('lm_router_topk_ws', (None, 0))]
