// Uploads in a row, each from the same host array that is overwritten as soon as
// the call returns, then downloads: every device array holds what it was sent.
// Arguments: page-locked buffers to be had, then sizes in bytes.
#include <algorithm>
#include <cstdio>

#include "../../akantu_amd/csrc/akx_copy.hpp"

int main(int argc, char** argv) {
  fake_pinned_left = std::atol(argv[1]);
  std::vector<size_t> sizes;
  for (int k = 2; k < argc; ++k) sizes.push_back(size_t(std::atoll(argv[k])));
  FakeStream stream;
  akx::HostCopier copy;
  size_t most = 1;
  for (size_t n : sizes) most = std::max(most, n);
  std::vector<unsigned char> host(most), back(most);
  auto value = [](size_t round, size_t k, size_t i) {
    return static_cast<unsigned char>(round * 101 + k * 37 + i * 7 + (i >> 12));
  };
  for (size_t round = 0; round < 3; ++round) {
    std::vector<std::vector<unsigned char>> dev;
    for (size_t n : sizes) dev.emplace_back(n);
    for (size_t k = 0; k < sizes.size(); ++k) {
      for (size_t i = 0; i < sizes[k]; ++i) host[i] = value(round, k, i);
      if (copy.to_device(0, &stream, dev[k].data(), host.data(), sizes[k])) return 2;
      std::memset(host.data(), 0, host.size());
    }
    for (size_t k = 0; k < sizes.size(); ++k) {
      if (copy.to_host(0, &stream, back.data(), dev[k].data(), sizes[k])) return 3;
      for (size_t i = 0; i < sizes[k]; ++i)
        if (back[i] != value(round, k, i)) {
          std::printf("round %zu array %zu byte %zu\n", round, k, i);
          return 1;
        }
    }
    if (hipStreamSynchronize(&stream)) return 4;
  }
  copy.release();
  return 0;
}
