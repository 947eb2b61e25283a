// Device helpers of the grouped (multi-job) launches: the next virtual blocks a
// workgroup takes, and the job that owns a virtual block.
// Included inside namespace apirl::(anonymous) of the kernel sources.
#ifndef APIRL_GROUP_COMMON_H
#define APIRL_GROUP_COMMON_H

// Virtual blocks are handed out `grab` at a time (the round header's, tuned per batch; 1 if
// unset): the first to a workgroup by its own number, the rest by a per-phase counter, so a
// workgroup that drew cheap blocks takes more (they differ ~10x in cost) and a round with no
// more than one draw per workgroup, or an empty phase, never touches the counter (2048
// workgroups drawing from it took 26 us).  A value >= total: no work left.
__device__ __forceinline__ int grab_size(const BatchHeader* hdr) {
  return hdr->grab > 0 ? hdr->grab : 1;
}
__device__ __forceinline__ long first_vb(int grab) { return (long)blockIdx.x * grab; }
__device__ __forceinline__ long next_vb(unsigned long long* ctr, int grab, long total) {
  __shared__ long s_vb;
  const long dealt = (long)gridDim.x * grab;
  if (dealt >= total) return total;
  __syncthreads();  // every lane has read the previous draw
  if (threadIdx.x == 0) s_vb = dealt + (long)atomicAdd(ctr, (unsigned long long)grab);
  __syncthreads();
  return s_vb;
}

// Last job whose first virtual block is <= vb (jobs are sorted by first).
template <class J>
__device__ __forceinline__ int find_job(const J* jobs, int n, long vb) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (jobs[mid].first <= vb) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

#endif
