// dsm.hpp -- what the two passes A of the dynamic Smagorinsky model
// (dsm_fused.hip in FP64, dsm_fp32.hip in FP32) share.
#pragma once
#include "kernels.hpp"

namespace chan {

// longest z chunk a block marches
constexpr int DSM_KMAX = 64;
// Cross-lane moves along x.  Columns are x-fastest with CX columns per row
// and CX divides the wave, so lane l's x neighbours are lanes l-1 and l+1; a
// whole-wave shift by one lane (DPP wave_shr:1 / wave_shl:1) delivers them.
// The ends of a row (halo columns, which produce no output) receive a lane of
// another row, or 0 at the ends of the wave.
// The whole wave must be active.
constexpr int DPP_WAVE_SHL1 = 0x130, DPP_WAVE_SHR1 = 0x138;
template <int CTRL>
__device__ inline double lane_shift(double v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (unsigned long long)(unsigned)lo | ((unsigned long long)(unsigned)hi << 32));
}
template <int CTRL>
__device__ inline float lane_shift(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// |S| of the unique cell of plane p <= nzp + 1 at byte offset `own` of the
// plane (column c) and of its periodic images: columns 1, nxg-1, nxg from
// nxg-2, 2, 3 and planes 1, nzg-1, nzg from nzg-2, 2, 3
template <typename T>
__device__ __forceinline__ void store_smag(T* smag, const Dims& d, int p, unsigned own, int c, T v)
{
    char* const S = (char*)(smag + (long)(p - 1) * d.sxy);
    *(T*)(S + own) = v;
    const int pz = p <= 3 ? p + d.nzp : (p == d.nzp + 1 ? 1 : 0);
    const int dx = c <= 3 ? d.nxp : (c == d.nxp + 1 ? -d.nxp : 0);
    const unsigned img = own + dx * (int)sizeof(T);
    if (dx) *(T*)(S + img) = v;
    if (pz) {
        char* const Sz = (char*)(smag + (long)(pz - 1) * d.sxy);
        *(T*)(Sz + own) = v;
        if (dx) *(T*)(Sz + img) = v;
    }
}

// The block's compute_dt maxima (m3: this lane's), per wave by a butterfly,
// then over the waves, into its slot of b.dtpart (one per block of the
// member's grid); wmax: LDS, one entry per wave
template <int NT, typename T>
__device__ __forceinline__ void dt_block_maxima(double (&m3)[3], double (*wmax)[3], int tid, const GBlk& gb,
                                                const DsmBufs<T>& b)
{
    for (int m = 32; m > 0; m >>= 1)
        for (int c = 0; c < 3; c++) m3[c] = fmax(m3[c], __shfl_xor(m3[c], m, 64));
    if ((tid & 63) == 0)
        for (int c = 0; c < 3; c++) wmax[tid >> 6][c] = m3[c];
    __syncthreads();
    if (tid < 3) {
        double v = 0.0;
        for (int w = 0; w < NT / 64; w++) v = fmax(v, wmax[w][tid]);
        const int nb = gb.gx * gb.gy * gb.gz;
        b.dtpart[(long)tid * nb + (gb.z * gb.gy + gb.y) * gb.gx + gb.x] = v;
    }
}

inline void dsm_check(int kchunk, int tile, int first)
{
    if (kchunk < 1 || kchunk > DSM_KMAX || tile < first || tile > 3) {
        fprintf(stderr, "chanles: DSM z chunk %d or tile %d out of range\n", kchunk, tile);
        abort();
    }
}

}  // namespace chan
