"""VeLO's launches by the number of tensors and blocks, at their edges and against the oracle: few blocks (the gradients' and the
LSTM's launches paired, ``k_velo_p0_feat``), with one tensor, without a matrix, with N-D tensors only, a vector of many rows of
sums, 256 tensors and one more; and many tensors (``k_velo_gates_many``, 64 tensors a block, and four rows a block in
``k_velo_heads``) at remainders of both, with numbers of unit blocks that do and do not divide among the XCDs.
"""

import pytest
import torch

from golden_io import max_err

pytestmark = pytest.mark.gpu

REL, ABS = 1e-5, 1e-6


def _small(n):
    return [[(3 + i % 5, 4 + i % 7), (5 + i % 9,), (2, 3, 1 + i % 3)][i % 3] for i in range(n)]


@pytest.mark.parametrize("shapes,hidden", [
    ([(33, 70)], 64), ([(64,), (1,), (4097,)], 128), ([(8, 4, 3, 3), (2, 3, 5, 14)], 64), ([(3000000,), (40, 300)], 64),
    ([(130, 260), (1, 513), (700, 3), (7,), (4, 1, 9)], 192), (_small(255), 64), (_small(256), 64), (_small(257), 64),
    (_small(767), 64), (_small(768), 64), (_small(769), 128), (_small(830), 256),
], ids=lambda v: str(len(v)) if isinstance(v, list) else "h%d" % v)
def test_follows_the_oracle(shapes, hidden):
    from oracle import pylo_oracle as O
    from pylo_amd import VeLO_CUDA
    from pylo_amd.models import VeLOMLP, VeLORNN

    torch.manual_seed(3)
    rnn = VeLORNN(lstm_hidden_size=hidden, param_inits=64)
    with torch.no_grad():
        rnn.lstm_init_state[0].normal_(0, 0.1)
        rnn.lstm_init_state[1].normal_(0, 0.1)
    mlp = VeLOMLP(param_inits=64)
    gen = torch.Generator().manual_seed(17)
    cpu = [torch.randn(s, generator=gen) * 0.3 for s in shapes]
    gpu = [torch.nn.Parameter(v.clone().cuda()) for v in cpu]
    kw = dict(lr=1e-2, num_steps=50, weight_decay=1e-3)
    orc = O.VeloOracle(cpu, rnn.state_dict(), mlp.state_dict(), **kw)
    opt = VeLO_CUDA(gpu, rnn=rnn, mlp=mlp, **kw)
    for t in range(4):
        grads = [torch.randn(s, generator=gen) * 10.0 ** (-(i % 4)) for i, s in enumerate(shapes)]
        for p, g in zip(gpu, grads):
            p.grad = g.cuda()
        loss = torch.tensor(1.5 - 0.2 * t)
        orc.step(grads, loss)
        opt.step(loss.cuda())
        checks = [("h", opt.lstm_hidden_state[0], orc.h), ("c", opt.lstm_hidden_state[1], orc.c)]
        checks += [(i, p, cpu[i]) for i, p in enumerate(gpu)]
        for tag, got, ref in checks:
            assert max_err(got, ref, REL, ABS) <= 1.0, (t, tag)
