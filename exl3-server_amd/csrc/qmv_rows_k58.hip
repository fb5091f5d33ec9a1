// k_qmv_rows for codebook widths K = 5..8 (templates in qmv_rows.hpp).
#include "qmv_rows.hpp"

namespace exl3h {

void launch_qmv_rows_k58(int K, int cb, int rb, int waves, const exl3d::RowsArgs &a, hipStream_t st) {
  switch (K) {
    case 5: qmv_rows_cb<5>(cb, rb, waves, a, st); break;
    case 6: qmv_rows_cb<6>(cb, rb, waves, a, st); break;
    case 7: qmv_rows_cb<7>(cb, rb, waves, a, st); break;
    default: qmv_rows_cb<8>(cb, rb, waves, a, st);
  }
}

}  // namespace exl3h
