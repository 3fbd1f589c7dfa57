// Instantiations of the output layer's kernels (lmhead.h) and their launcher.
#include "launchers.h"
#include "lmhead.h"

namespace fie {

template <int DT, int WM, int WN>
static void tile_of(const uint16_t* h, const uint16_t* w, uint16_t* out, const KParams& P, int H, int wide,
                    hipStream_t st)
{
    constexpr int BM = 64 * WM, BN = 64 * WN;
    const int nrb = (P.a.rows + BM - 1) / BM, tiles = (P.a.vocab + BN - 1) / BN;
    k_lmhead_tile<DT, WM, WN><<<8 * ((tiles + 7) / 8) * nrb, 64 * WM * WN, 0, st>>>(
        h, w, out, P.a.row_stride, P.a.rows, P.a.vocab, H, nrb, wide);
}

template <int DT>
static void lmhead_dt(const KParams& P, const void* hidden, const void* weight, int H, hipStream_t st)
{
    const uint16_t* h = (const uint16_t*)hidden;
    const uint16_t* w = (const uint16_t*)weight;
    uint16_t* out = (uint16_t*)P.a.logits;
    const int wide = ((uintptr_t)out % 8) == 0 && P.a.row_stride % 4 == 0;
    const int B = P.a.rows;
    // the least rows that hold the batch up to 128 (a row of a tile left over is work
    // for nothing), then two 128-row blocks beside each other; figures in lmhead.h
    if (B <= 64) tile_of<DT, 1, 4>(h, w, out, P, H, wide, st);
    else if (B <= 128) tile_of<DT, 2, 2>(h, w, out, P, H, wide, st);
    else tile_of<DT, 2, 4>(h, w, out, P, H, wide, st);
}

hipError_t launch_lmhead(const KParams& P, const void* hidden, const void* weight, int H, hipStream_t st)
{
    if (P.a.dtype == FIE_F16) lmhead_dt<FIE_F16>(P, hidden, weight, H, st);
    else lmhead_dt<FIE_BF16>(P, hidden, weight, H, st);
    return hipGetLastError();
}

}  // namespace fie
