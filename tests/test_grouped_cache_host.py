"""A grouped segment that the table marks as kept in the cache is read with plain loads in
every SELL layout, one that is not with non-temporal loads, and a pass that reads a matrix
once keeps nothing: run on the CPU, where non-temporal loads are counted."""
import pytest

from host_kernels import build, device_part, run

MAIN = r"""
using namespace mife;
using namespace mife::grouped;
int main(int, char** argv) {
  // a diagonal matrix of 130 rows in three slices (node rows: 43 in one), one column each
  const int kind = std::atoi(argv[1]), keep = std::atoi(argv[2]), once = std::atoi(argv[3]);
  const bool nodes = kind == 2;
  const int rows = nodes ? 129 : 130, ns = nodes ? 1 : 3;
  std::vector<int> rp(ns + 1), col(64 * ns), cb(ns, 0);
  std::vector<uint16_t> c16(64 * ns);
  std::vector<double> val((nodes ? 9 : 1) * 64 * ns, 0.0), x(256, 1.0), y(256, 0.0);
  for (int s = 0; s <= ns; ++s) rp[s] = 64 * s;
  for (int k = 0; k < 64 * ns; ++k) {
    const int c = std::min(k, (nodes ? rows / 3 : rows) - 1);
    col[k] = c16[k] = c;
    if (nodes) for (int d = 0; d < 3; ++d) val[4 * d * 64 + k] = 2.0;
    else val[k] = 2.0;
  }
  mife_segment S{};
  S.n = rows;
  S.format = nodes ? MIFE_FMT_SELL3 : MIFE_FMT_SELL;
  S.n_slices = ns;
  S.cb_off = kind == 0 ? -1 : 0;
  View V{};
  V.rp = rp.data(), V.col = col.data(), V.col16 = c16.data(), V.cbase = cb.data();
  Block B{0, 0, ns, 0, 0, 1, keep, kUpdateBlocks};
  emu::launch(1, 256, [&] {
    auto f = [&](int row, double ax) { y[row] = ax; };
    NoHook none;
    if (once) block_rows<double>(V, B, S, val.data(), x.data(), f);
    else block_walk<double>(V, B, S, val.data(), x.data(), [](int) { return 0; },
                            [&](int row, double ax, int) { f(row, ax); }, none);
  });
  int wrong = 0;
  for (int i = 0; i < rows; ++i) wrong += y[i] != 2.0;
  std::printf("%ld %d\n", emu::streamed_loads, wrong);
}
"""


@pytest.fixture(scope="module")
def grouped(tmp_path_factory):
    source = device_part("mife_grouped.hip", "using namespace mife;\nusing namespace mife::grouped;", "")
    return build(tmp_path_factory.mktemp("grouped"), source, MAIN)


@pytest.mark.parametrize("kind", [0, 1, 2], ids=["sell32", "sell16", "sell3"])
@pytest.mark.parametrize("keep,once", [(1, 0), (0, 0), (1, 1)])
def test_kept_segments_take_plain_loads(grouped, kind, keep, once):
    streamed, wrong = run(grouped, kind, keep, once)
    assert wrong == 0
    loads = 64 * 10 if kind == 2 else 2 * 192  # every value and column once
    assert streamed == (loads if once or not keep else 0)
