// Launch planning of the class kernels: what jk_launch.hip needs of the
// translation units that hold the kernels.
#pragma once
#include "jk_class_kernels.h"

enum { GEN_JK = 0, GEN_IP1 = 1 };

// Third argument of the gradient and runtime-l kernels.
struct GenExtra {
    double *ejk;        // natm x 3 (gradient mode)
    double jf, kf;      // factors of the J and K parts of the two-particle density
};

// Survival predicate of the energy-gradient contraction
// (gpu4pyscf/lib/gvhf-rys/create_tasks.cu:858-877), float32 in the same order.
__device__ __forceinline__ bool survives_ejk(float q_kl, float kl_cutoff, uint32_t bas_ij,
                                             uint32_t bas_kl, int ish, int jsh, int nbas,
                                             const float *dc, bool do_j, bool do_k)
{
    if (!(q_kl >= kl_cutoff && bas_ij >= bas_kl)) return false;
    const int ksh = bas_kl / nbas, lsh = bas_kl - (bas_kl / nbas) * nbas;
    const float d_cutoff = kl_cutoff - q_kl;
    return (do_k && (dc[ish*nbas+lsh] + dc[jsh*nbas+ksh] > d_cutoff ||
                     dc[ish*nbas+ksh] + dc[jsh*nbas+lsh] > d_cutoff)) ||
           (do_j && dc[bas_ij] + dc[bas_kl] > d_cutoff);
}

// classes with a shell of l >= 4, and the energy gradients of large classes:
// the runtime-l kernels of jk_generic.hip (GEN_TB threads).  Plan of one task:
// kl_chunk of d, workgroups, dynamic LDS in bytes; false for an unsupported
// class.
#define GEN_TB          256
bool jk_generic_plan(const JKTask &k, int mode, TaskDesc &d, long &blocks, size_t &lds);
const void *jk_generic_kernel_of(int mode);

// the per-lane gradient kernel of a class (key: li*125 + lj*25 + lk*5 + ll),
// one wavefront per workgroup, or NULL (jk_ip1.hip)
const void *jk_ip1_lane_kernel_of(int key);

// What a run of class tasks computes: J/K (GEN_JK) or the energy gradient.
struct JKRun {
    int mode;
    GenExtra ex;
};

// Launches `ntasks` validated tasks; a supplies the fields they share.
hipError_t jk_launch_tasks(const JKBuildArgs &a, const JKTask *tasks, int ntasks,
                           void *const *streams, int nstreams, const JKRun &run);

// The launches that jk_launch_tasks would make (jk_plan_tasks): the first nmax
// items into out, their number into n.
hipError_t jk_plan_launches(const JKBuildArgs &a, const JKTask *tasks, int ntasks,
                            const JKRun &run, JKPlanItem *out, int nmax, int &n);
