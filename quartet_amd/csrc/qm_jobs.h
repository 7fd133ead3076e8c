// Job kernels.  A job is the work of one kernel launch as a struct: its arguments, `blocks` (how many 256-thread
// workgroups it needs) and `run(block)`, the body of one workgroup.  `job_kernel` runs one job or
// several independent ones in a single grid, the first job's blocks first: the next job's blocks fill the machine
// while the first one drains, and the pause between two dependent launches of a stream is paid once.
//
// Wave priorities.  A job's workgroup computes its addresses, requests its input, works on it for a few thousand
// vector instructions and stores.  Eight such waves share a SIMD, and left alone they move in step: a new wave's few
// dozen address instructions queue behind seven neighbours' arithmetic, its loads go out late, and memory idles while
// the arithmetic runs and the reverse.  A job kernel therefore starts at the highest wave priority and the job calls
// job_requests_issued() once its loads are out (back to the lowest), so that a fresh wave's requests overtake the
// running waves' arithmetic.  Measured on several MI355X: forward quantizer of 8192 x 4096 19.4 -> 17.4-18.3 us,
// stochastic-rounding quantizer -4 to -6 %, inverse rotation -3 %, transposing and re-quantizing kernels -1 to -2 %;
// on two slower-clocked chips of the pool the forward quantizer was unchanged and the others gained the same.
// Priorities order waves of one SIMD only; results do not depend on them.
#pragma once
#include <hip/hip_runtime.h>

namespace qm {

__device__ __forceinline__ void job_starts() { __builtin_amdgcn_s_setprio(3); }
__device__ __forceinline__ void job_requests_issued() { __builtin_amdgcn_s_setprio(0); }
// before the final stores: a wave that is about to leave makes room for the next one sooner
__device__ __forceinline__ void job_stores_next() { __builtin_amdgcn_s_setprio(3); }

// Workgroup scratch of a job: dynamic LDS, sized for the largest job of the launch (J::kLds bytes).  As a static array in
// each job's body, two jobs of one kernel would be given the sum of their needs.
extern __shared__ uint4 job_lds[];

template <class A, class... Rest>
__device__ __forceinline__ void run_job(unsigned bid, const A& a, const Rest&... rest) {
    if constexpr (sizeof...(Rest) == 0) {
        a.run(bid);
    } else {
        if (bid < a.blocks) a.run(bid);
        else run_job(bid - a.blocks, rest...);
    }
}

// J::kWaves: resident waves per SIMD the job is to be compiled for (1: the fewest it can do with, 0: what the launch's other jobs
// want), for the job of a launch that wants fewest
template <typename... Ts>
constexpr int wanted_waves(Ts... waves) {
    int least = 0;
    ((least = waves && (!least || waves < least) ? waves : least), ...);
    return least ? least : 1;
}

template <class... Jobs>
__global__ __launch_bounds__(256, wanted_waves(Jobs::kWaves...)) void job_kernel(Jobs... jobs) {
    job_starts();
    run_job(blockIdx.x, jobs...);
}

// independent jobs in one grid, the first job's blocks first
template <class... Jobs>
void launch_jobs(hipStream_t stream, const Jobs&... jobs) {
    unsigned lds = 0;
    ((lds = (unsigned)Jobs::kLds > lds ? (unsigned)Jobs::kLds : lds), ...);
    job_kernel<Jobs...><<<dim3((jobs.blocks + ...)), dim3(256), lds, stream>>>(jobs...);
}
template <class A>
void launch_job(const A& job, hipStream_t stream) {
    launch_jobs(stream, job);
}

}  // namespace qm
