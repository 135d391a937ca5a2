"""Every barrier of the MINRES kernels is reached by all threads of a block, also in the
launch that finds the solve finished, whatever number of wavefronts shares a slice; run
on the CPU, with the solution checked."""
import pytest

from host_kernels import build, device_part, run

MAIN = r"""
using namespace mife;
int main(int, char** argv) {
  const int split = std::atoi(argv[1]), limit = std::atoi(argv[2]);
  // symmetric indefinite tridiagonal matrix, scheduled SELL of three slices, int32 columns
  const int n = 150, ns = 3, span = sell_order_span(ns);
  std::vector<int> ptr(ns + 1), col;
  std::vector<double> val, b(n), x(n, 0.0), want(n);
  auto a = [&](int i, int j) { return i == j ? (i % 2 ? -3.0 : 4.0) : 1.0; };
  for (int s = 0; s < ns; ++s) {
    ptr[s] = (int)col.size();
    for (int j = -1; j <= 1; ++j)
      for (int l = 0; l < 64; ++l) {
        const int i = 64 * s + l, c = i + j;
        const bool in = i < n && c >= 0 && c < n;
        col.push_back(in ? c : std::min(i, n - 1));
        val.push_back(in ? a(i, c) : 0.0);
      }
  }
  ptr[ns] = (int)col.size();
  std::vector<int4> order(8 * span, int4{-1, 0, 0, 0});
  for (int s = 0; s < ns; ++s) order[s * span] = int4{s, ptr[s], 3, 0};
  for (int i = 0; i < n; ++i) want[i] = std::sin(i + 1.0);
  for (int i = 0; i < n; ++i) {
    b[i] = 0;
    for (int c = std::max(0, i - 1); c <= std::min(n - 1, i + 1); ++c) b[i] += a(i, c) * want[c];
  }
  MatArgs A{n, MIFE_FMT_SELL, ptr.data(), col.data(), ns, nullptr, (const int32_t*)order.data(), span, split, 16, 16};
  std::vector<double> dinv(n), r1(n), r2(n), z(n), w(n), w2(n), v(n, 0.0), t(n);
  for (int i = 0; i < n; ++i) dinv[i] = 1.0 / std::abs(a(i, i));
  static MinresState st;
  const int grid = 8, vg = (n + 255) / 256;
  emu::launch(grid, 256, [&] {
    minres_init_kernel<MIFE_FMT_SELL, 64, double>(A, val.data(), b.data(), x.data(), dinv.data(), r1.data(), r2.data(),
                                                  z.data(), w.data(), w2.data(), &st, 1e-9, limit);
  });
  int k = 0;
  for (; k < 500 && !st.s[k & 1].done; ++k) {
    emu::launch(grid, 256, [&] {
      minres_a_kernel<MIFE_FMT_SELL, 64, double>(A, val.data(), z.data(), v.data(), t.data(), r1.data(), w.data(),
                                                 w2.data(), x.data(), &st, k, k == 0 ? grid : vg);
    });
    emu::launch(vg, 256, [&] {
      minres_b_kernel(n, t.data(), r1.data(), r2.data(), z.data(), dinv.data(), &st, k, grid);
    });
  }
  double err = 0;
  for (int i = 0; i < n; ++i) err = std::max(err, std::abs(x[i] - want[i]));
  std::printf("%ld %d %.3e\n", emu::partial_barriers, st.s[k & 1].iters, err);
  return 0;
}
"""


@pytest.fixture(scope="module")
def minres(tmp_path_factory):
    return build(tmp_path_factory.mktemp("minres"), device_part("mife_krylov.hip"), MAIN)


@pytest.mark.parametrize("split,limit", [(1, 400), (2, 400), (4, 400), (4, 3), (4, 0)])
def test_minres_barriers_are_reached_by_whole_blocks(minres, split, limit):
    partial, iters, err = run(minres, split, limit)
    assert partial == 0
    assert iters == limit if limit < 400 else iters < 400
    if limit == 400:  # residual fallen by 1e9, condition number below 10
        assert err <= 1e-7
