"""The LM step at the edges of its blocks: one free parameter, odd counts,
counts beside multiples of the 2 x 4 blocks of the normal matrix, the most that fit LDS,
and response columns of 1e33 times the usual size, whose squares leave the range that the first
pass assumes.  Checks and tolerances are those of test_lm_step_vs_oracle."""
import pytest

from test_gpu_lm import test_lm_step_vs_oracle as step_vs_oracle

pytestmark = pytest.mark.gpu

SIZES = [{"T": 1}, {"T": 2}, {"T": 3}, {"T": 4, "vz": 1}, {"T": 4, "Bz": 3}, {"T": 4, "Bz": 2, "vz": 3},
         {"T": 8, "Bz": 4, "vz": 5}, {"T": 16, "Bz": 9, "vz": 8}, {"T": 32, "Bz": 16, "vz": 15},
         {"T": 32, "Bz": 16, "vz": 16}]


@pytest.mark.parametrize("nodes", SIZES, ids=[str(sum(n.values())) for n in SIZES])
def test_sizes(gpu_ctx, cpu, nodes):
    step_vs_oracle(gpu_ctx, cpu, nodes, 1, None)


class Scaled:
    """A context whose responses of one free parameter are scaled."""

    def __init__(self, ctx, j, f):
        self.__dict__.update(ctx=ctx, j=j, f=f)

    def __getattr__(self, name):
        return getattr(self.ctx, name)

    def forward_nodes_torch(self, atm):
        st, eqv, status = self.ctx.forward_nodes_torch(atm)
        eqv[:, self.j] *= self.f
        return st, eqv, status


@pytest.mark.parametrize("j", [0, 2, 4])
def test_large_responses(gpu_ctx, cpu, j):
    step_vs_oracle(Scaled(gpu_ctx, j, 1e33), cpu, {"T": 3, "vz": 2}, 1, None)
