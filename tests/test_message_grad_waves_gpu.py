"""Edge gradients of the message kernels at every block size of their dispatch (4, 8 and 16 waves):
receivers with no edge, with fewer edges than the block has waves, and with many rounds of edges for each
wave and one more for some, against the oracle's autograd in float64."""
import pytest
import torch

from conftest import assert_rel
from oracle.tensor_product import TensorProductOracle
from test_message_gpu import _edge_inputs, _op

pytestmark = pytest.mark.gpu


# up to two blocks per CU (512 receivers of one chunk on 256 CUs), up to 32 and above, and the waves there
@pytest.mark.parametrize("lmax,receivers,harmonics,waves", [
    (2, 8200, True, 4), (1, 8200, True, 4), (2, 8200, False, 8), (2, 530, True, 8), (2, 530, False, 8),
    (3, 530, True, 8), (3, 530, False, 8), (2, 20, True, 16), (3, 20, True, 16),
    (3, 20, False, 16)])
def test_edge_gradients(gpu, lmax, receivers, harmonics, waves):
    c = 40                                           # a ragged chunk: lanes past the channels
    many = 64 * waves + waves // 2 + 1               # a last round of edges in some waves only
    counts = torch.arange(receivers) % 3             # 0, 1, 2 edges
    counts[1] = many
    counts[-1] = waves + 1
    generator = torch.Generator().manual_seed(receivers + lmax)
    dst = torch.repeat_interleave(torch.arange(receivers), counts)
    dst = dst[torch.randperm(len(dst), generator=generator)]
    src = torch.randint(0, receivers, (len(dst),), generator=generator)
    op = _op(c, lmax, lmax, lmax, gpu)
    ref = TensorProductOracle(c, lmax, lmax, lmax)
    inputs = _edge_inputs(ref, receivers, len(dst), 5)
    go = torch.randn(receivers, ref.output_width, generator=generator)
    wanted = (0, 1, 2) if harmonics else (0, 2)
    dev = [t.to(gpu).requires_grad_(i in wanted) for i, t in enumerate(inputs)]
    cpu = [t.double().requires_grad_(i in wanted) for i, t in enumerate(inputs)]
    out = op(*dev, src.to(gpu), dst.to(gpu))
    expect = ref.graph_message(*cpu, src, dst, edge_chunk_size=512)
    grads = torch.autograd.grad(out, [dev[i] for i in wanted], go.to(gpu), create_graph=True)
    egrads = torch.autograd.grad(expect, [cpu[i] for i in wanted], go.double(), create_graph=True)
    for i, a, b in zip(wanted, grads, egrads):
        assert_rel(a, b, what=f"gradient {i}, {waves} waves")
    # the tangent kernels, through the second derivatives
    probe = [torch.randn(t.shape, generator=generator) for t in grads]
    second = torch.autograd.grad(grads, [dev[i] for i in wanted], [p.to(gpu) for p in probe])
    esecond = torch.autograd.grad(egrads, [cpu[i] for i in wanted], [p.double() for p in probe])
    for i, a, b in zip(wanted, second, esecond):
        assert_rel(a, b, what=f"second derivative {i}, {waves} waves")
