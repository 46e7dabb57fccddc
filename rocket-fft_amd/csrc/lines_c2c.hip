// lines_c2c.hip -- the general line kernel: plain complex lines and the four-step passes.
#include "mixlaunch.hpp"

namespace rfh {

template <typename T>
void launch_mix_c2c(int op, const dev::LineArgs<T> &a, const MixGeom &m, hipStream_t s) {
  switch (op) {
    case dev::OP_C2C: launch_mix_op<T, dev::OP_C2C>(a, m, s); break;
    case dev::OP_PASSA: launch_mix_op<T, dev::OP_PASSA>(a, m, s); break;
    case dev::OP_PASSB: launch_mix_op<T, dev::OP_PASSB>(a, m, s); break;
    default: RFH_THROW(1, "internal error: no line kernel for op " + std::to_string(op));
  }
}

template void launch_mix_c2c<float>(int, const dev::LineArgs<float> &, const MixGeom &, hipStream_t);
template void launch_mix_c2c<double>(int, const dev::LineArgs<double> &, const MixGeom &, hipStream_t);

}  // namespace rfh
