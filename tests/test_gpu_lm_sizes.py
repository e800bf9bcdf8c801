"""The LM step at the edges of its blocks: one free parameter, odd counts,
counts beside multiples of the 2 x 4 blocks of the normal matrix, the most that fit LDS;
response columns above the 1e30 beyond which their sums are formed, and columns whose sum
passes REAL(4).  Checks and tolerances are those of test_lm_step_vs_oracle."""
import numpy as np
import pytest

from test_gpu_lm import NOISE, problem
from test_gpu_lm import _delta_err as delta_err, _model_err as model_err, _oracle_step as oracle_step
from test_gpu_lm import test_lm_step_vs_oracle as step_vs_oracle

pytestmark = pytest.mark.gpu

SIZES = [{"T": 1}, {"T": 2}, {"T": 3}, {"T": 4, "vz": 1}, {"T": 4, "Bz": 3}, {"T": 4, "Bz": 2, "vz": 3},
         {"T": 8, "Bz": 4, "vz": 5}, {"T": 16, "Bz": 9, "vz": 8}, {"T": 32, "Bz": 16, "vz": 15},
         {"T": 32, "Bz": 16, "vz": 16}]


@pytest.mark.parametrize("nodes", SIZES, ids=[str(sum(n.values())) for n in SIZES])
def test_sizes(gpu_ctx, cpu, nodes):
    step_vs_oracle(gpu_ctx, cpu, nodes, 1, None)


class Edited:
    """A context whose responses an edit changes in place."""

    def __init__(self, ctx, edit):
        self.__dict__.update(ctx=ctx, edit=edit)

    def __getattr__(self, name):
        return getattr(self.ctx, name)

    def forward_nodes_torch(self, atm):
        st, eqv, status = self.ctx.forward_nodes_torch(atm)
        self.edit(eqv)
        return st, eqv, status


FLT_MAX = float(np.finfo(np.float32).max)
BIG = {"T": 32, "Bz": 16, "vz": 17}       # work arrays in device memory


@pytest.mark.parametrize("nodes,js", [({"T": 3, "vz": 2}, (0,)), ({"T": 3, "vz": 2}, (2, 4)), (BIG, (20, 60))],
                         ids=["first", "two", "big"])
def test_large_responses(gpu_ctx, cpu, nodes, js):
    """Columns of up to 1e32: their sums are formed, none overflows."""

    def edit(eqv):
        for j in js:
            m = eqv[:, j].abs().amax(dim=1, keepdim=True)
            assert float(m.min()) > 0
            eqv[:, j] = eqv[:, j] / m * 1e32
            assert float(eqv[:, j].abs().amax(dim=1).min()) > 1e30
            assert float(eqv[:, j].abs().double().sum(dim=1).max()) < FLT_MAX

    step_vs_oracle(Edited(gpu_ctx, edit), cpu, nodes, 1, None)


# 448 rows of one value: below and above the largest sum, by 1 %
@pytest.mark.parametrize("value,over", [(7.5e35, False), (7.67e35, True), (1e37, True)])
@pytest.mark.parametrize("nodes,j", [({"T": 3, "vz": 2}, 0), ({"T": 3, "vz": 2}, 3), ({"T": 32, "Bz": 16, "vz": 16}, 20),
                                     (BIG, 0), (BIG, 64)], ids=["5-0", "5-3", "64-20", "big-0", "big-64"])
def test_columns_whose_sum_overflows_are_zeroed(gpu_ctx, cpu, nodes, j, value, over):
    """In every second pixel one column's absolute sum passes REAL(4): it is
    zero in the step and in the best response functions, the others and the
    other pixels stay as they are (forward.f90:672-678)."""
    import torch
    P = problem(gpu_ctx, cpu, nodes, nx=2, ny=2)
    ncol, nf, numw = P["ncol"], P["nfreq"], P["numw"]
    assert nf == 448 and (nf * value > FLT_MAX) == over and value > 1e30
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()       # noqa: E731
    atm = d(P["guess"].astype(np.float32))
    st, eqv, _ = gpu_ctx.forward_nodes_torch(atm)
    eqv[::2, j] = torch.where(eqv[::2, j] < 0, -value, value)
    h_eqv, h_cur = eqv.cpu().numpy(), atm.cpu().numpy()
    ref_eqv = h_eqv.copy()
    if over:
        ref_eqv[::2, j] = 0.0
    sla = np.tile(np.array([0, 1e29, 1e29, 0, 0, 0, 0, 0, 10.0]), (ncol, 1))
    bsyn, ebest, best = torch.zeros((ncol, nf), dtype=torch.float64, device="cuda"), torch.ones_like(eqv), atm.clone()
    delta = torch.zeros((ncol, P["ifreep"]), dtype=torch.float64, device="cuda")
    isig = np.full(nf, 1.0 / NOISE ** 2)
    ref = oracle_step(cpu, P, P["obs"], st.cpu().numpy().reshape(ncol, 4 * numw).astype(np.float64),
                      np.zeros((ncol, nf)), sla, ref_eqv, np.zeros_like(h_eqv), isig, h_cur, h_cur)
    gpu_ctx.lm_step_torch(d(P["obs"]), st, bsyn, d(sla), eqv, ebest, d(isig), atm, best, delta=delta)
    torch.cuda.synchronize()
    assert np.array_equal(ebest.cpu().numpy(), ref_eqv)
    g_del, g_cur = delta.cpu().numpy(), atm.cpu().numpy()
    for c in range(ncol):
        assert delta_err(g_del[c], ref[c][5]) <= 1e-6 and model_err(g_cur, c, ref[c][0]) <= 2e-6
