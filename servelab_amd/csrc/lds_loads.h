// Loads that go from global memory straight into LDS (global_load_lds_dwordx4): a wavefront's 64 loads of 16
// bytes land side by side in 1 KB at `lds_at`.  They pass the registers by, so the compiler neither counts
// nor waits for them: wait_loads<N> returns once at most the N youngest loads of the wavefront are under way, and
// its reads of LDS are done: behind the barrier that follows, another wavefront's loads may land where they read (the
// compiler moves products of the last reads, and the wait for these with them, behind a barrier).
// (M0 holds the place in LDS; a load that reads it may not follow the instruction that writes it without a wait state between.)
#pragma once
__device__ __forceinline__ void load_to_lds(const void* from, unsigned lds_at) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(from), "s"(lds_at) : "m0");
}
// The same from a base that all lanes share and an offset of the lane's own.
__device__ __forceinline__ void load_to_lds(unsigned offset, const void* base, unsigned lds_at) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" : : "v"(offset), "s"(lds_at), "s"(base) : "m0");
}
template <int N_> __device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_s_waitcnt((N_ & 15) | (7 << 4) | ((N_ >> 4) << 14));
}
// Rows of 128 bytes in LDS, eight units of 16 bytes each: unit c of row r lies at place c ^ lds_place(r), so that the 16
// lanes that read unit c of rows r .. r + 15 touch 16 different 16-byte slots of a 256-byte line of banks, and each half of
// them 8 different slots of a 128-byte one.
__device__ __forceinline__ int lds_place(int r) { return ((r >> 1) & 7) ^ (4 * (r & 1)); }
// The lane's number, worked out where it stands: kept in no register through a loop that has none to spare.
__device__ __forceinline__ int lane_here() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(l));
  return l;
}
