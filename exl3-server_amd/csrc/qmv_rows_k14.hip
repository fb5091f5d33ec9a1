// k_qmv_rows for codebook widths K = 1..4 (templates in qmv_rows.hpp).
#include "qmv_rows.hpp"

namespace exl3h {

void launch_qmv_rows_k14(int K, int cb, int rb, int waves, const exl3d::RowsArgs &a, hipStream_t st) {
  switch (K) {
    case 1: qmv_rows_cb<1>(cb, rb, waves, a, st); break;
    case 2: qmv_rows_cb<2>(cb, rb, waves, a, st); break;
    case 3: qmv_rows_cb<3>(cb, rb, waves, a, st); break;
    default: qmv_rows_cb<4>(cb, rb, waves, a, st);
  }
}

}  // namespace exl3h
