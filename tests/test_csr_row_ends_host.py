"""Back-substitution and the lifted RHS on rows that end at the last int32 entry index
(2^31 - 1): the kernels run on the CPU, with the entry arrays placed so that only those
rows exist and any signed overflow trapped, against plain sums."""
import pytest

from host_kernels import build, definition, run

MAIN = r"""
using namespace mife;
int main(int, char** argv) {
  // rows of `len` entries, the last one ending at 2^31 - 1
  const int n = std::atoi(argv[1]), len = std::atoi(argv[2]), compat = std::atoi(argv[3]);
  const long long total = (long long)n * len, first = 2147483647LL - total;
  std::vector<int> rp(n + 1), col(total), free_idx(n), new_idx(n);
  std::vector<double> val(total), u(std::max(n, len)), src(n), rhs(n), R(n), b(n);
  for (int i = 0; i <= n; ++i) rp[i] = (int)(first + (long long)i * len);
  for (long long k = 0; k < total; ++k) col[k] = (int)((7 * k + 3) % n), val[k] = std::sin(k + 1.0);
  for (size_t i = 0; i < u.size(); ++i) u[i] = std::cos(3.0 * i);
  for (int i = 0; i < n; ++i) free_idx[i] = i, new_idx[i] = i % 3 ? i : -1, src[i] = 0.5 * i, rhs[i] = 1.0 / (i + 1);
  const int* colp = (const int*)((uintptr_t)col.data() - (uintptr_t)first * sizeof(int));
  const double* valp = (const double*)((uintptr_t)val.data() - (uintptr_t)first * sizeof(double));
  BACKSUB
  emu::launch((n + kRhsRows - 1) / kRhsRows, 256, [&] {
    solver_rhs_kernel(n, free_idx.data(), rp.data(), colp, valp, new_idx.data(), u.data(), src.data(), rhs.data(),
                      nullptr, b.data());
  });
  double err = 0;
  for (int i = 0; i < n; ++i) {
    double r = -src[i], v = src[i] + rhs[i];
    for (int j = 0; j < len; ++j) {
      const long long k = (long long)i * len + j;
      r += val[k] * u[compat ? j : col[k]];
      if (new_idx[col[k]] < 0) v -= val[k] * u[col[k]];
    }
    err = std::max(err, std::max(std::abs(R[i] - r), std::abs(b[i] - v)));
  }
  std::printf("%.3e\n", err);
  return 0;
}
"""
BACKSUB = """const int rows = std::atoi(argv[4]);
  auto back = [&](auto r, auto c) {
    constexpr int ROWS = decltype(r)::value;
    emu::launch((n + ROWS - 1) / ROWS, 256, [&] {
      backsub_kernel<ROWS, decltype(c)::value>(n, rp.data(), colp, valp, u.data(), src.data(), nullptr, R.data());
    });
  };
  auto pick = [&](auto r) { compat ? back(r, std::true_type{}) : back(r, std::false_type{}); };
  if (rows == 16) pick(std::integral_constant<int, 16>{});
  else pick(std::integral_constant<int, 32>{});"""


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    parts = ["kRhsRows", "solver_rhs_kernel", "kBsTile", "backsub_kernel"]
    source = '#include "mife_sparse.hpp"\nnamespace mife {\n' + "".join(definition("mife_sparse.hip", p) for p in parts)
    return build(tmp_path_factory.mktemp("rows"), source + "}\n", MAIN.replace("BACKSUB", BACKSUB), "-ftrapv")


@pytest.mark.parametrize("compat", [0, 1])
@pytest.mark.parametrize("block_rows", [16, 32])
@pytest.mark.parametrize("n,len_", [(1, 5), (3, 70), (33, 61), (40, 130), (2, 5000)])
def test_rows_at_the_end_of_the_index_range(rows, n, len_, block_rows, compat):
    err, = run(rows, n, len_, compat, block_rows, timeout=20)
    assert err <= 1e-15 * (len_ + 2) * (len_ + n)  # rows of len_ products below 1
