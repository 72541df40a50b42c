// The device-wide scan of csrc/blockscan.hpp on the host, one block after the
// other in an order of dispatch given by the caller: each block runs to its end
// before the next one begins, so a block that waits for one not yet begun never
// ends.  scan_progress ROWS N ORDER (0 forward, 1 backward, else a seed)
#include <algorithm>
#include <numeric>
#include <random>

#include "../../gpucelllistsph.jl_amd/csrc/blockscan.hpp"

using namespace gclsph;

namespace {
std::vector<int32_t> items;
std::vector<int32_t> out32;
std::vector<int64_t> out64;
std::vector<uint64_t> words;
int32_t largest = 0;
int64_t n = 0;

template <int Rows>
void starts() {
  scan_tile<Rows, true>(items.data(), out32.data(), n, words.data(), &largest);
}
template <int Rows>
void offsets() {
  scan_tile<Rows, false>(items.data(), out64.data(), n, words.data(), nullptr);
}

template <int Rows>
int check(int64_t order) {
  const int64_t tiles = scan_tiles(n, Rows);
  std::vector<unsigned> dispatch(static_cast<size_t>(tiles));
  std::iota(dispatch.begin(), dispatch.end(), 0u);
  if (order == 1) std::reverse(dispatch.begin(), dispatch.end());
  if (order > 1) std::shuffle(dispatch.begin(), dispatch.end(), std::mt19937_64(uint64_t(order)));
  gridDim.x = unsigned(tiles);
  std::mt19937_64 rng(7);
  items.resize(size_t(n));
  for (auto& v : items) v = int32_t(rng() % 5);
  std::vector<int64_t> sum(size_t(n) + 1, 0);
  std::partial_sum(items.begin(), items.end(), sum.begin() + 1, [](int64_t a, int64_t b) { return a + b; });
  const int32_t top = *std::max_element(items.begin(), items.end());
  out64.assign(size_t(n) + 1, -1);
  out32.assign(size_t(n) + 1, -1);
  for (auto f : {&offsets<Rows>, &starts<Rows>}) {
    words.assign(size_t(scan_words(n)), ~uint64_t(0));
    for (int64_t i = 0; i < 512; ++i) clear_scan_words(words.data(), n, i, 512);
    for (unsigned b : dispatch) {
      blockIdx.x = b;
      block::run(kScanThreads, f);
    }
  }
  if (!std::equal(sum.begin(), sum.end(), out64.begin()) || !std::equal(sum.begin(), sum.end(), out32.begin()) ||
      largest != top || std::any_of(items.begin(), items.end(), [](int32_t v) { return v != 0; })) {
    std::printf("wrong sums\n");
    return 1;
  }
  return 0;
}
}  // namespace

int main(int, char** argv) {
  const int rows = std::atoi(argv[1]);
  n = std::atoll(argv[2]);
  const int64_t order = std::atoll(argv[3]);
  return rows == 4 ? check<4>(order) : rows == 8 ? check<8>(order) : check<16>(order);
}
