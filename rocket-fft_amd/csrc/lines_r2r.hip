// lines_r2r.hip -- the general line kernel: real-to-real lines (DCT, DST, Hartley, FFTPACK).
#include "mixlaunch.hpp"

namespace rfh {

template <typename T>
void launch_mix_r2r(int op, const dev::LineArgs<T> &a, const MixGeom &m, hipStream_t s) {
  switch (op) {
    case dev::OP_R2R: launch_mix_op<T, dev::OP_R2R>(a, m, s); break;
    default: RFH_THROW(1, "internal error: no line kernel for op " + std::to_string(op));
  }
}

template void launch_mix_r2r<float>(int, const dev::LineArgs<float> &, const MixGeom &, hipStream_t);
template void launch_mix_r2r<double>(int, const dev::LineArgs<double> &, const MixGeom &, hipStream_t);

}  // namespace rfh
