// lines_blue.hip -- the general line kernel: Bluestein lines and rows.
#include "mixlaunch.hpp"

namespace rfh {

template <typename T>
void launch_mix_blue(int op, const dev::LineArgs<T> &a, const MixGeom &m, hipStream_t s) {
  switch (op) {
    case dev::OP_BLUE: launch_mix_op<T, dev::OP_BLUE>(a, m, s); break;
    case dev::OP_BLUEROW: launch_mix_op<T, dev::OP_BLUEROW>(a, m, s); break;
    default: RFH_THROW(1, "internal error: no line kernel for op " + std::to_string(op));
  }
}

template void launch_mix_blue<float>(int, const dev::LineArgs<float> &, const MixGeom &, hipStream_t);
template void launch_mix_blue<double>(int, const dev::LineArgs<double> &, const MixGeom &, hipStream_t);

}  // namespace rfh
