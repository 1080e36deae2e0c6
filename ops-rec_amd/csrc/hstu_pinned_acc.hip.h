// Matrix accumulators in fixed registers: block n of 32 x 32 sums is a[16 n] .. a[16 n + 15] of the accumulator half of the register
// file, named in assembly.  Left to itself the compiler has all 32x32 results of a kernel either in accumulators -- and then copies
// every score out to the vector registers before it can compute on it, 16 instructions a block -- or in vector registers, where the
// output sums then leave no room for the operands.  Here the sums stay in the accumulators throughout and only the scores pass
// through vector registers (the source is compiled with the matrix instructions' results in vector registers, see _build.py).
//
// The compiler does not know what these registers hold.  It would use them for values of its own only when it is out of vector
// registers; acc_fence() keeps any such value from living across it, and stands in every phase of the kernels.  Nor does it know what
// the assembly here needs: that the vector unit leaves an operand of acc_mfma() alone for two instructions ahead of it, and that nobody
// touches the registers of a load in assembly before its wait.  tests/test_host_pinned_registers.py looks for all three in what the
// compiler makes of the kernels that use this header.
#pragma once
#include <utility>

#include "hstu_fwd_kernel.hip.h"

namespace hstu {

// Nothing the compiler keeps in the first REGS accumulators lives across this.
template <int REGS>
__device__ __forceinline__ void acc_fence()
{
    static_assert(REGS == 64 || REGS == 128 || REGS == 256, "lists exist for these");
#define HSTU_ACC_64 \
    "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", "a16",       \
    "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", "a32",    \
    "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", "a48",    \
    "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63"           
#define HSTU_ACC_128 HSTU_ACC_64, \
    "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79",    \
    "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95",    \
    "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109",        \
    "a110", "a111", "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123",    \
    "a124", "a125", "a126", "a127"                                                                                    
#define HSTU_ACC_256 HSTU_ACC_128, \
    "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141",    \
    "a142", "a143", "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155",    \
    "a156", "a157", "a158", "a159", "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169",    \
    "a170", "a171", "a172", "a173", "a174", "a175", "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183",    \
    "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191", "a192", "a193", "a194", "a195", "a196", "a197",    \
    "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", "a208", "a209", "a210", "a211",    \
    "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223", "a224", "a225",    \
    "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239",    \
    "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253",    \
    "a254", "a255"                                                                                                    
    if constexpr (REGS == 64) {
        asm volatile("" ::: HSTU_ACC_64);
    } else if constexpr (REGS == 128) {
        asm volatile("" ::: HSTU_ACC_128);
    } else {
        asm volatile("" ::: HSTU_ACC_256);
    }
#undef HSTU_ACC_64
#undef HSTU_ACC_128
#undef HSTU_ACC_256
}

// block N += A . B.  (An operand that the vector unit has just written is ready: two instructions later at the latest, which the
// callers' schedules give it.)
template <typename Tag, int N>
__device__ __forceinline__ void acc_mfma(u32x4_t a, u32x4_t b)
{
    if constexpr (std::is_same<Tag, bf16_tag>::value) {
        asm volatile("v_mfma_f32_32x32x16_bf16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), "n"(16 * N), "n"(16 * N + 15));
    } else {
        asm volatile("v_mfma_f32_32x32x16_f16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), "n"(16 * N), "n"(16 * N + 15));
    }
}
template <int I>
__device__ __forceinline__ float acc_read()
{
    float x;
    asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(I));
    return x;
}
template <int I>
__device__ __forceinline__ void acc_zero()
{
    asm volatile("v_accvgpr_write_b32 a[%0], 0" ::"n"(I));
}
// registers 0 .. sizeof...(I) - 1
template <int... I>
__device__ __forceinline__ void acc_zero_all(std::integer_sequence<int, I...>)
{
    (acc_zero<I>(), ...);
}
// waits until the last products have written their sums
__device__ __forceinline__ void acc_settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }
template <int N, int... I>
__device__ __forceinline__ f32x16_t acc_block(std::integer_sequence<int, I...>)
{
    const f32x16_t r = {acc_read<16 * N + I>()...};
    return r;
}
// f(0), f(1), .. f(N - 1) with compile-time arguments
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

}  // namespace hstu
