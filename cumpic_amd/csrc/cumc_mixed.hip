// cumc_mixed.hip -- FP32 instantiations of the reconstruction, Riemann and EMF kernels (the
// mixed-precision form).  Built separately from cumc.hip so that these kernels may contract
// multiply-adds and use the hardware FP32 reciprocal / square root, while the FP64 drop-in
// path keeps every operation separately rounded.  The conserved state, the RK3 combination,
// the conserved-to-primitive recovery and the face-B update stay FP64 (k_tail).
#include "ctx.hpp"

void stage_mixed(cumc_ctx *ctx, int st, bool comb) { stage<float>(ctx, ctx->F32, st, comb); }

// the reference's ghost passes (and torus inflow clamps) on the FP32 primitive planes
void launch_ghost32(cumc_ctx *ctx, int st)
{
    const Lay &L = ctx->L;
    const Fields<float> &G = ctx->F32;
    hipLaunchKernelGGL(k_ghost<float>, dim3(nblk(ghost_threads(L), 256)), dim3(256), 0, ctx->stream, L, G.P32, G.EPS32,
                       G.BC32, ctx->M, ctx->dt_dev, st, ctx->dt_pub);
}

void fluxes_mixed(cumc_ctx *ctx, int dir, double *aos_tmp)
{
    const Lay &L = ctx->L;
    const long ncell = (long)(L.nx + 6) * (L.ny + 6) * (L.nz + 6);
    launch_fluxes<float>(ctx, ctx->F32, dir);
    hipLaunchKernelGGL((k_flux_to_aos<float>), dim3(nblk(ncell, 256)), dim3(256), 0, ctx->stream, L,
                       ctx->F32.F[dir - 1], aos_tmp);
}
