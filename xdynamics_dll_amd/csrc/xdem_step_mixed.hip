// xdem_step_mixed.hip -- mixed-precision instantiation of the fused step kernels:
// contact-force arithmetic and the neighbours' velocity copies in FP32; the pair test,
// positions, tangential history, force sums and the Verlet update in FP64.
#include <algorithm>

#include "xdem_step.hpp"

namespace xdem {
namespace {

constexpr unsigned kBlock = 256;
inline dim3 grid_for(unsigned n) { return dim3((n + kBlock - 1) / kBlock); }

// pass 0: the lite pass over every sphere outside this step's full pass (two kernels in
// fused mode); pass 2: the triangle pass (meshes), before pass 1, the full pass over the
// spheres k_touch queued. The full-pass kernels stride over the queue segments (the queue
// lengths are on the device) with A.full_blocks blocks, a multiple of kQueueSegs. The two
// passes touch disjoint spheres and may run concurrently.
// per_block: the fewest spheres worth a block.
inline dim3 full_grid(const StepArgs& A, unsigned per_block)
{
    const unsigned blocks = (A.np + per_block - 1) / per_block;
    return dim3((std::min(A.full_blocks, std::max(blocks, 1u)) + kQueueSegs - 1) / kQueueSegs * kQueueSegs);
}

template <bool MULTI, bool FUSE, int MODEL, bool GPU_LAW>
void collide_passes(const StepArgs& A, int pass, hipStream_t s)
{
    const dim3 g = grid_for(A.np), b(kBlock);
    if (pass == 1) {
        if (A.has_cyl) hipLaunchKernelGGL((k_collide<float, MULTI, FUSE, MODEL, GPU_LAW, true>), full_grid(A, 4), b, 0, s, A);
        else hipLaunchKernelGGL((k_collide<float, MULTI, FUSE, MODEL, GPU_LAW, false>), full_grid(A, 4), b, 0, s, A);
    } else if (pass == 2) {
        // the triangle pass (grid-strided over the mesh queue, whose length is on the device)
        hipLaunchKernelGGL((k_mesh_pass<float, MULTI, MODEL, GPU_LAW>), full_grid(A, kBlock), b, 0, s, A);
    } else if (FUSE) {
        launch_lite_fused(A, MULTI, s);
    } else {
        hipLaunchKernelGGL((k_collide_lite<float, MULTI, false, MODEL, GPU_LAW>), g, b, 0, s, A);
    }
}

template <bool MULTI, bool FUSE>
void collide_models(const StepArgs& A, int model, bool gpu_law, int pass, hipStream_t s)
{
    if (model == 1) {
        if (gpu_law) collide_passes<MULTI, FUSE, 1, true>(A, pass, s);
        else collide_passes<MULTI, FUSE, 1, false>(A, pass, s);
    } else {
        if (gpu_law) collide_passes<MULTI, FUSE, 0, true>(A, pass, s);
        else collide_passes<MULTI, FUSE, 0, false>(A, pass, s);
    }
}

hipError_t collide_mixed(const StepArgs& A, bool multi, bool fuse, int model, bool gpu_law, int pass,
                         hipStream_t s)
{
    if (A.np == 0) return hipSuccess;
    if (multi) {
        if (fuse) collide_models<true, true>(A, model, gpu_law, pass, s);
        else collide_models<true, false>(A, model, gpu_law, pass, s);
    } else {
        if (fuse) collide_models<false, true>(A, model, gpu_law, pass, s);
        else collide_models<false, false>(A, model, gpu_law, pass, s);
    }
    return hipGetLastError();
}

}  // namespace

CollideLaunch collide_launch_mixed() { return collide_mixed; }

}  // namespace xdem
