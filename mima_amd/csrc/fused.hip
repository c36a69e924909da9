// The band phase of the one-pass forward+backward of both sides in one
// persistent kernel (FP32): LW and SW work items from one counter.  No
// counterpart in the reference.  The per-unit arithmetic is that of the LW
// LDS-table backward kernel and of the SW backward band kernel
// (lw_vjp_body.hpp, sw_vjp_body.hpp); what changes is the schedule: one launch
// whose workgroups move from LW items to SW items without a kernel boundary,
// instead of two kernels on two streams.  Measured at 131072 x 60, before the LW
// body took several g-points a lane, it was the slower schedule (88.1 against
// 81.2 ms per forward+backward step): the SW body's registers hold the shared
// kernel at two waves per SIMD.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "lw_vjp_body.hpp"
#include "rrtmg_device.hpp"
#include "sw_vjp_body.hpp"

namespace rrtmg {

size_t fused_lds_bytes(const LwLdsPlan &plan, int sw_nlay)
{
    return std::max((size_t)plan.fwd_lds_bytes, (size_t)FUSED_WGW * sw_vjp_lds_bytes(sw_nlay, sizeof(float)));
}

size_t fused_row_floats(int lw_nlay, int sw_nlay)
{
    return std::max(lw_vjp_row_bytes(lw_nlay, sizeof(float), LWV_LDS), sw_vjp_state_bytes(sw_nlay, sizeof(float))) / sizeof(float);
}

int fused_grid(const LwLdsPlan &plan, int nitems) { return std::min(plan.ncu, nitems); }

// the SW body is a call of its own, so that its registers do not weigh on the LW
// body's; the LW arithmetic has the same bits wherever it is compiled
// (lw_rows.hpp)

// 8 waves per workgroup at up to 256 VGPRs: two waves per SIMD
__global__ __launch_bounds__(64 * FUSED_WGW) __attribute__((amdgpu_waves_per_eu(2)))
void fused_band_kernel(FusedBand a)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float *lds = (float *)smem_raw;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    float *row = a.rows + ((size_t)blockIdx.x * FUSED_WGW + wave) * a.row_floats;
    float *ktab = (float *)(smem_raw + LW_ET_VECS * 16);
    const size_t sw_wave_lds = sw_vjp_lds_bytes(a.sin.nlay, sizeof(float)) / sizeof(float);
    __shared__ int s_item;
    const SwUnitArgs<float> sa = sw_unit_args<float>(a.sin, a.sw, a.sexp_off, a.stab);
    const LwUnitArgs la = lw_unit_args(a.lin, a.lw, a.plk_off, a.ltab, a.cst);
    int loaded = -1;  // the LW band whose k-tables LDS holds
    for (;;) {
        // (next_item synchronises the workgroup: every wave is done with the
        // previous item, and with what it kept in LDS, before the next starts)
        const int item = next_item(a.items, &s_item);
        if (item >= a.nitems) break;
        if (item < a.litems) {
            const int tile = item / LW_TILE_ITEMS;
            const LwTileSlot slot = LW_TILE_SLOTS.s[item - tile * LW_TILE_ITEMS];
            const int b = slot.band - 1;
            if (loaded < 0)  // a workgroup's first item: the LW items come before the SW ones
                for (int i = threadIdx.x; i < LW_ET_VECS; i += 64 * FUSED_WGW)
                    ((uint4 *)smem_raw)[i] = ((const uint4 *)(a.ltab + a.et_off))[i];
            if (b != loaded) {
                lw_copy_tables(ktab, a.ltab, a.plan, b);
                __syncthreads();
                loaded = b;
            }
            const int cend = min((tile + 1) * LW_TILE, a.lin.ncol);
            for (int k = wave; k < 16; k += FUSED_WGW) {
                const int c0 = tile * LW_TILE + (slot.part * 16 + k) * slot.cpw;
                if (c0 >= cend) break;
                lw_vjp_unit_of(la, a.lbands, b, (lptr<const ExpTfn<float>>)smem_raw, (lptr<const float>)ktab, c0, cend,
                               lane, (gptr<float>)row);
            }
        } else {
            loaded = -1;  // the SW units' LDS overlays the LW tables
            const int blk = (item - a.litems) * FUSED_WGW + wave;
            if (blk >= a.snunits) continue;
            const int tile = blk / a.snwaves;
            const WaveUnit u = a.sunits[blk % a.snwaves];
            const SwBand B = a.sbands[u.band];
            float *smem = lds + (size_t)wave * sw_wave_lds;
#define SBODY(jb)                                                                                  \
    case jb - 16:                                                                                  \
        sw_vjp_unit<jb, float>(sa, B, u, tile, lane, (gptr<float>)row, (lptr<float>)smem);       \
        break;
            switch (u.band) { SW_BANDS(SBODY) }
#undef SBODY
        }
    }
}

hipError_t launch_fused_band(const FusedBand &a, hipStream_t s)
{
    hipLaunchKernelGGL(reset_items_kernel, dim3(1), dim3(1), 0, s, a.items);
    hipLaunchKernelGGL(fused_band_kernel, dim3(fused_grid(a.plan, a.nitems)), dim3(64 * FUSED_WGW),
                       fused_lds_bytes(a.plan, a.sin.nlay), s, a);
    return hipGetLastError();
}

}  // namespace rrtmg
