// lines_real.hip -- the general line kernel: real lines to half spectra and back.
#include "mixlaunch.hpp"

namespace rfh {

template <typename T>
void launch_mix_real(int op, const dev::LineArgs<T> &a, const MixGeom &m, hipStream_t s) {
  switch (op) {
    case dev::OP_R2C_EVEN: launch_mix_op<T, dev::OP_R2C_EVEN>(a, m, s); break;
    case dev::OP_R2C_ODD: launch_mix_op<T, dev::OP_R2C_ODD>(a, m, s); break;
    case dev::OP_C2R_EVEN: launch_mix_op<T, dev::OP_C2R_EVEN>(a, m, s); break;
    case dev::OP_C2R_ODD: launch_mix_op<T, dev::OP_C2R_ODD>(a, m, s); break;
    default: RFH_THROW(1, "internal error: no line kernel for op " + std::to_string(op));
  }
}

template void launch_mix_real<float>(int, const dev::LineArgs<float> &, const MixGeom &, hipStream_t);
template void launch_mix_real<double>(int, const dev::LineArgs<double> &, const MixGeom &, hipStream_t);

}  // namespace rfh
