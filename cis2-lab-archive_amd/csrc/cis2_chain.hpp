// cis2_chain.hpp — the strict left-to-right chain over LDS groups that the
// persistent decode kernel, the lone GEMV and the few-row GEMM share.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cis2 {
namespace {

// acc + the floats of 16 * npair groups (16 bytes, ST groups apart, the group
// address per lane), strictly in order, as one assembly loop over two fixed sets of 8
// groups (v[192:223], v[224:255]): the next set's 8 reads go out, one wait
// for the current set (issued a set earlier), its 32 adds.  Left to the
// compiler, the same loop inside the decode kernel kept the sum or the
// loop address in a register of the set read last and drained the reads
// (lgkmcnt(0)) once or twice per 64 adds: 8 to 10 cycles per add against
// 6.1 here (MI355X, one wave, 4096 adds).  The block starts with a full
// drain, so the counts inside are exact (LDS reads return in order); it
// reads 8 groups past the range (never added: the caller keeps that LDS
// readable) and drains them before the registers are released.  The adds
// are the same IEEE adds in the same order and operand order.  npair >= 1,
// wave-uniform.
#define CIS2_LD(R0, R3, K, BASE) \
  "ds_read_b128 v[" #R0 ":" #R3 "], %[ad] offset:" BASE "+" #K "*%[s]\n\t"
#define CIS2_ADD4(A, B, C, D)                                                   \
  "v_add_f32 %[acc], v" #A ", %[acc]\n\tv_add_f32 %[acc], v" #B ", %[acc]\n\t" \
  "v_add_f32 %[acc], v" #C ", %[acc]\n\tv_add_f32 %[acc], v" #D ", %[acc]\n\t"
#define CIS2_SET_A(BASE) CIS2_LD(192, 195, 0, BASE) CIS2_LD(196, 199, 1, BASE) CIS2_LD(200, 203, 2, BASE) CIS2_LD(204, 207, 3, BASE) CIS2_LD(208, 211, 4, BASE) CIS2_LD(212, 215, 5, BASE) CIS2_LD(216, 219, 6, BASE) CIS2_LD(220, 223, 7, BASE)
#define CIS2_SET_B(BASE) CIS2_LD(224, 227, 0, BASE) CIS2_LD(228, 231, 1, BASE) CIS2_LD(232, 235, 2, BASE) CIS2_LD(236, 239, 3, BASE) CIS2_LD(240, 243, 4, BASE) CIS2_LD(244, 247, 5, BASE) CIS2_LD(248, 251, 6, BASE) CIS2_LD(252, 255, 7, BASE)
#define CIS2_ADDS_A CIS2_ADD4(192, 193, 194, 195) CIS2_ADD4(196, 197, 198, 199) CIS2_ADD4(200, 201, 202, 203) CIS2_ADD4(204, 205, 206, 207) CIS2_ADD4(208, 209, 210, 211) CIS2_ADD4(212, 213, 214, 215) CIS2_ADD4(216, 217, 218, 219) CIS2_ADD4(220, 221, 222, 223)
#define CIS2_ADDS_B CIS2_ADD4(224, 225, 226, 227) CIS2_ADD4(228, 229, 230, 231) CIS2_ADD4(232, 233, 234, 235) CIS2_ADD4(236, 237, 238, 239) CIS2_ADD4(240, 241, 242, 243) CIS2_ADD4(244, 245, 246, 247) CIS2_ADD4(248, 249, 250, 251) CIS2_ADD4(252, 253, 254, 255)
#define CIS2_CLOB "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199", "v200", "v201", "v202", "v203", "v204", "v205", "v206", "v207", "v208", "v209", "v210", "v211", "v212", "v213", "v214", "v215", "v216", "v217", "v218", "v219", "v220", "v221", "v222", "v223", "v224", "v225", "v226", "v227", "v228", "v229", "v230", "v231", "v232", "v233", "v234", "v235", "v236", "v237", "v238", "v239", "v240", "v241", "v242", "v243", "v244", "v245", "v246", "v247", "v248", "v249", "v250", "v251", "v252", "v253", "v254", "v255"
template <uint32_t ST>
__device__ __forceinline__ float chain_lds16(const __attribute__((address_space(3))) void* p, uint32_t npair, float acc) {
  uint32_t ad = (uint32_t)(uintptr_t)p;
  asm volatile(
      "s_waitcnt lgkmcnt(0)\n\t" CIS2_SET_A("0")
      "1:\n\t" CIS2_SET_B("8*%[s]")
      "s_waitcnt lgkmcnt(8)\n\t" CIS2_ADDS_A
      "v_add_u32 %[ad], 16*%[s], %[ad]\n\t" CIS2_SET_A("0")
      "s_waitcnt lgkmcnt(8)\n\t" CIS2_ADDS_B
      "s_sub_u32 %[n], %[n], 1\n\t"
      "s_cmp_lg_u32 %[n], 0\n\t"
      "s_cbranch_scc1 1b\n\t"
      "s_waitcnt lgkmcnt(0)"
      : [acc] "+v"(acc), [ad] "+v"(ad), [n] "+s"(npair)
      : [s] "i"(ST * 16)
      : "memory", "scc", CIS2_CLOB);
  return acc;
}
// chain_lds16 over v[96:127] and v[128:159], for kernels that keep three waves
// per SIMD (at most 168 registers).
#define CIS2_RSET_A(BASE) CIS2_LD(96, 99, 0, BASE) CIS2_LD(100, 103, 1, BASE) CIS2_LD(104, 107, 2, BASE) CIS2_LD(108, 111, 3, BASE) CIS2_LD(112, 115, 4, BASE) CIS2_LD(116, 119, 5, BASE) CIS2_LD(120, 123, 6, BASE) CIS2_LD(124, 127, 7, BASE)
#define CIS2_RSET_B(BASE) CIS2_LD(128, 131, 0, BASE) CIS2_LD(132, 135, 1, BASE) CIS2_LD(136, 139, 2, BASE) CIS2_LD(140, 143, 3, BASE) CIS2_LD(144, 147, 4, BASE) CIS2_LD(148, 151, 5, BASE) CIS2_LD(152, 155, 6, BASE) CIS2_LD(156, 159, 7, BASE)
#define CIS2_RADDS_A CIS2_ADD4(96, 97, 98, 99) CIS2_ADD4(100, 101, 102, 103) CIS2_ADD4(104, 105, 106, 107) CIS2_ADD4(108, 109, 110, 111) CIS2_ADD4(112, 113, 114, 115) CIS2_ADD4(116, 117, 118, 119) CIS2_ADD4(120, 121, 122, 123) CIS2_ADD4(124, 125, 126, 127)
#define CIS2_RADDS_B CIS2_ADD4(128, 129, 130, 131) CIS2_ADD4(132, 133, 134, 135) CIS2_ADD4(136, 137, 138, 139) CIS2_ADD4(140, 141, 142, 143) CIS2_ADD4(144, 145, 146, 147) CIS2_ADD4(148, 149, 150, 151) CIS2_ADD4(152, 153, 154, 155) CIS2_ADD4(156, 157, 158, 159)
#define CIS2_RCLOB "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", "v109", "v110", "v111", "v112", "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125", "v126", "v127", "v128", "v129", "v130", "v131", "v132", "v133", "v134", "v135", "v136", "v137", "v138", "v139", "v140", "v141", "v142", "v143", "v144", "v145", "v146", "v147", "v148", "v149", "v150", "v151", "v152", "v153", "v154", "v155", "v156", "v157", "v158", "v159"
template <uint32_t ST>
__device__ __forceinline__ float chain_lds16_low(const __attribute__((address_space(3))) void* p, uint32_t npair, float acc) {
  uint32_t ad = (uint32_t)(uintptr_t)p;
  asm volatile(
      "s_waitcnt lgkmcnt(0)\n\t" CIS2_RSET_A("0")
      "1:\n\t" CIS2_RSET_B("8*%[s]")
      "s_waitcnt lgkmcnt(8)\n\t" CIS2_RADDS_A
      "v_add_u32 %[ad], 16*%[s], %[ad]\n\t" CIS2_RSET_A("0")
      "s_waitcnt lgkmcnt(8)\n\t" CIS2_RADDS_B
      "s_sub_u32 %[n], %[n], 1\n\t"
      "s_cmp_lg_u32 %[n], 0\n\t"
      "s_cbranch_scc1 1b\n\t"
      "s_waitcnt lgkmcnt(0)"
      : [acc] "+v"(acc), [ad] "+v"(ad), [n] "+s"(npair)
      : [s] "i"(ST * 16)
      : "memory", "scc", CIS2_RCLOB);
  return acc;
}

// The same loop over a ring of four slots of 16 groups (1 KiB apart, 64 KiB
// at LDS address `ring`, a multiple of 64 KiB) that other waves fill: slots
// 0 .. nslot-1 in turn, slot i at ring + (i % 4) * 16 KiB, the lane's group at
// ad in slot 0.  Slot i is complete once every wave has passed barrier i: the
// caller has passed barrier 0, the loop passes barriers 1 .. nslot-1, each
// just before the first reads of its slot go out.  Those reads, and the ones
// in flight across a barrier, are of slots i and i+1, so the others may write
// slot i+2 after barrier i+1.  Its sets are chain_lds16_low's.  nslot >= 1, wave-uniform.
__device__ __forceinline__ float chain_ring(uint32_t ad, uint32_t ring, uint32_t nslot, float acc) {
  uint32_t n = nslot - 1;
  const uint32_t mask = 0xffffu;
  asm volatile(
      "s_waitcnt lgkmcnt(0)\n\t" CIS2_RSET_A("0")
      "s_cmp_eq_u32 %[n], 0\n\t"
      "s_cbranch_scc1 2f\n\t"
      "1:\n\t" CIS2_RSET_B("8*%[s]")
      "s_waitcnt lgkmcnt(8)\n\t" CIS2_RADDS_A
      "v_add_u32 %[ad], 16*%[s], %[ad]\n\t"
      "v_and_or_b32 %[ad], %[ad], %[mask], %[ring]\n\t"
      "s_barrier\n\t" CIS2_RSET_A("0")
      "s_waitcnt lgkmcnt(8)\n\t" CIS2_RADDS_B
      "s_sub_u32 %[n], %[n], 1\n\t"
      "s_cmp_lg_u32 %[n], 0\n\t"
      "s_cbranch_scc1 1b\n\t"
      "2:\n\t" CIS2_RSET_B("8*%[s]")
      "s_waitcnt lgkmcnt(8)\n\t" CIS2_RADDS_A
      "s_waitcnt lgkmcnt(0)\n\t" CIS2_RADDS_B
      // early clobbers: acc, ad and n change before ring and mask are last read
      : [acc] "+&v"(acc), [ad] "+&v"(ad), [n] "+&s"(n)
      : [s] "i"(1024), [ring] "v"(ring), [mask] "s"(mask)
      : "memory", "scc", CIS2_RCLOB);
  return acc;
}
#undef CIS2_RSET_A
#undef CIS2_RSET_B
#undef CIS2_RADDS_A
#undef CIS2_RADDS_B
#undef CIS2_RCLOB
#undef CIS2_CLOB
#undef CIS2_LD
#undef CIS2_ADD4
#undef CIS2_SET_A
#undef CIS2_SET_B
#undef CIS2_ADDS_A
#undef CIS2_ADDS_B

}  // namespace
}  // namespace cis2
