// rows.hip — launches of the batched decode step's matrix kernels (rows.hpp).
#include "rows.hpp"
#include "internal.hpp"

using namespace pocr;

namespace {

template <int QT, int EPI, int NS>
void launch_rows(hipStream_t s, const RowsParams &p) {
    const int blocks = p.rows / 16;
    const dim3 threads(kRowsThreads);
    if (p.ntok <= kRowsPackMax) {
        hipLaunchKernelGGL((k_rows<QT, EPI, NS, true, 16>), dim3(blocks), threads, 0, s, p);
        return;
    }
    if constexpr (EPI == R_OPROJ || EPI == R_DOWN) {
        // a workgroup reads its whole operand image (295 KB at 3,072 columns
        // and 16 rows) at a CU's L2 rate: two halves where that leaves half the
        // chip idle
        if (p.ntok > 8 && blocks <= 128) {
            hipLaunchKernelGGL((k_rows<QT, EPI, NS, false, 8>), dim3(blocks, 2), threads, 0, s, p);
            return;
        }
    }
    hipLaunchKernelGGL((k_rows<QT, EPI, NS, false, 16>), dim3(blocks), threads, 0, s, p);
}

template <int QT>
int launch_rows_epi(hipStream_t s, int epi, const RowsParams &p) {
    switch (epi) {
    case R_PLAIN: launch_rows<QT, R_PLAIN, 1>(s, p); break;
    case R_SWIGLU: launch_rows<QT, R_SWIGLU, 1>(s, p); break;
    case R_OPROJ: launch_rows<QT, R_OPROJ, 2>(s, p); break;
    default: launch_rows<QT, R_DOWN, 3>(s, p); break;
    }
    HIP_TRY(hipGetLastError());
    return POCR_OK;
}

}  // namespace

int pocr::rows_gemm(hipStream_t s, int qtype, int epi, const RowsParams &p) {
    if (p.ntok < 1 || p.ntok > kMaxBatch || p.rows % 16) return fail(POCR_ERR_UNSUPPORTED, "rows: %d of %d", p.ntok, p.rows);
    switch (qtype) {
    case QT_Q8: return launch_rows_epi<QT_Q8>(s, epi, p);
    case QT_Q4: return launch_rows_epi<QT_Q4>(s, epi, p);
    case QT_Q6: return launch_rows_epi<QT_Q6>(s, epi, p);
    default: return fail(POCR_ERR_UNSUPPORTED, "rows: qtype %d", qtype);
    }
}
