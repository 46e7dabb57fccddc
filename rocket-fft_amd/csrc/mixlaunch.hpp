// mixlaunch.hpp -- launch of the general line kernel (mixline.hpp) for one
// operation; each of lines_*.hip instantiates a few operations.
#pragma once

#include <mutex>
#include <set>
#include <string>
#include <utility>

#include "mixline.hpp"
#include "passes.hpp"

namespace rfh {

// Lines of one small butterfly, bound by the loads a CU keeps in flight, which
// are as short as the lines: the general form's registers (every radix to 17)
// allow five waves per SIMD (complex128: three), this one eight for most
// operations.  us, general -> this: 3 complex64 along axis 0 of 1.4M lines 26.6
// -> 20.8, rows of 3 27.4 -> 18.2, real lines of 3 along axis 0 of 2.8M 42.8 ->
// 29.9, of 2 lines (DCT-II) of 4.2M 105.6 -> 77.5.
constexpr int kShortThreads = 512;

// Waves per SIMD that the compiler is held to (1: what the threads allow).  Five
// for the sums of many complex64 lines with a prime: 29 of 144631 lines 33.6 us at
// four, 30.9 at five.  Six for complex64 groups that move flat, by three registers:
// r2c of 24 on 349525 lines 25.2 -> 21.3, 64M pairs of reals in lines of 48 332 -> 311.
constexpr int kernel_waves(bool dbl, int op, int form) {
  if (dbl) return 1;
  if (form == dev::kFlat) return 6;
  return form == dev::kPrime && op != dev::OP_PASSA ? 5 : 1;
}

template <typename T, int OP, int FORM>
__global__ void __launch_bounds__(FORM == 0 || FORM & dev::kPrime ? dev::kMixThreads<T>
                                                                  : kShortThreads,
                                  kernel_waves(sizeof(T) == 8, OP, FORM))
    k_lines(const dev::LineArgs<T> a, const MixGeom m, int64_t tile0) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  dev::mix_body<T, OP, FORM>(a, m, tile0 + int64_t(dev::xcd_tile()), smem_raw);
}

template <typename T, int OP>
void launch_mix_op(const dev::LineArgs<T> &a, const MixGeom &m, hipStream_t s) {
  const size_t lds = size_t(m.L * m.ld + m.ngen) * 2 * sizeof(T);
  const int64_t groups = (a.nlines + m.L - 1) / m.L;
  const int threads = (m.L * m.T + 63) / 64 * 64;
  if (threads > dev::kMixThreads<T> || lds > lds_limit())
    RFH_THROW(3, "line group of " + std::to_string(a.f.n) + " needs " + std::to_string(threads) +
                     " threads and " + std::to_string(lds) + " B of LDS");
  auto *fn = &k_lines<T, OP, 0>;
  if constexpr (!dev::is_blue_op(OP))
    if (!few_pairs(m)) fn = &k_lines<T, OP, dev::kPrime>;
  if constexpr (dev::is_flat_op(OP))
    if (threads <= kShortThreads && lds <= 65536) {
      if (m.flat && !(m.ngen && few_pairs(m)))
        fn = short_lines(m) ? &k_lines<T, OP, dev::kShort | dev::kFlat>
             : m.ngen       ? &k_lines<T, OP, dev::kFlat | dev::kPrime>
                            : &k_lines<T, OP, dev::kFlat>;
      else if (short_lines(m))
        fn = &k_lines<T, OP, dev::kShort>;
    }
  if constexpr (OP == dev::OP_R2R)
    if (a.sub & dev::R2R_SINCOS) fn = &k_lines<T, OP, dev::kPrime | dev::kSinCos>;
  if (lds > 65536) {  // raise the kernel's dynamic-LDS ceiling once per device
    static std::mutex mu;
    static std::set<std::pair<int, const void *>> done;
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    const void *f = reinterpret_cast<const void *>(fn);
    std::lock_guard<std::mutex> lk(mu);
    if (!done.count({dev, f})) {
      HIP_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    int(lds_limit())));
      done.insert({dev, f});
    }
  }
  for_launches(groups, threads, [&](int64_t first, int64_t count) {
    hipLaunchKernelGGL(fn, dim3(unsigned(count)), dim3(unsigned(threads)), lds, s, a, m, first);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
      RFH_THROW(2, std::string("line kernel launch (") + std::to_string(count) + " groups, " +
                       std::to_string(lds) + " B LDS, op " + std::to_string(OP) +
                       "): " + hipGetErrorString(e));
  });
}

}  // namespace rfh
