"""The part of a solver matrix that products read through the Infinity Cache (sixteenths
of its slices): what an iteration's vectors leave of it, on the CPU."""
import pytest

from host_kernels import build, run

MAIN = r"""
int main(int, char** argv) {
  std::printf("%d\n", mife::keep_sixteenths(std::atof(argv[1]) * 1e6, std::atof(argv[2]) * 1e6));
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    return build(tmp_path_factory.mktemp("rule"), '#include "mife_sparse.hpp"\n', MAIN)


@pytest.mark.parametrize("matrix,vectors,kept", [
    (0, 0, 16), (210, 0, 16), (211, 0, 15), (420, 0, 8), (3400, 0, 0),  # 210 MB at most
    (200, 20, 16), (200, 30, 16), (200, 31, 15),  # 230 MB with the vectors
    (192, 179, 4), (581, 224, 0),  # a Krylov basis that takes most of it, and nearly all
    (90, 248, 0), (90, 1e6, 0),  # vectors alone beyond it
])
def test_vectors_come_before_the_matrix(rule, matrix, vectors, kept):
    assert run(rule, matrix, vectors) == [kept]
