// Shared device helpers for librandumb_hip: Squirrel5 noise, bf16 conversion, MFMA fragments, errors.
// gfx950 only.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/randumb_hip.h"

namespace rdb {

// ----------------------------------------------------------------------------------------------- errors
int set_error(int code, const char *fmt, ...);  // records the message for rdb_last_error_string, returns code
int check_launch(const char *what);             // hipGetLastError -> positive code + message
int reserve_lds(const void *kernel, size_t smem, const char *name);  // dynamic-LDS limit of a kernel, set once per device

// ----------------------------------------------------------------------------------------------- noise
// Squirrel5 constants and the row/column mixing prime (reference: src/rten_cpp/RandumbTensor.py:140-145,
// src/rten_cpp/csrc/cuda/rten.cu:13-18).
constexpr uint32_t SQ5_N1 = 0xd2a80a3fu;
constexpr uint32_t SQ5_N2 = 0xa884f197u;
constexpr uint32_t SQ5_N3 = 0x6C736F4Bu;
constexpr uint32_t SQ5_N4 = 0xB79F3ABBu;
constexpr uint32_t SQ5_N5 = 0x1b56c4f5u;
constexpr uint32_t PRIME = 198491317u;
// (PRIME*n + m)*N1 + seed == n*PN1 + m*N1 + seed (mod 2^32): lets a loop over n or m advance the first
// round with one add instead of a multiply.
constexpr uint32_t PN1 = (uint32_t)((uint64_t)PRIME * (uint64_t)SQ5_N1);

// Rounds after "b = idx*N1 + seed" (reference: RandumbTensor.py:151-159).
__device__ __forceinline__ uint32_t sq5_tail(uint32_t b)
{
    b ^= (b >> 9);
    b += SQ5_N2;
    b ^= (b >> 11);
    b *= SQ5_N3;
    b ^= (b >> 13);
    b += SQ5_N4;
    b ^= (b >> 15);
    b *= SQ5_N5;
    b ^= (b >> 17);
    return b;
}

// The same for kernels that do nothing but hash, a value at a time: exclusive ors that the compiler cannot merge with the additions that follow into v_xad_u32
// (one instruction that issues alone, below).  69 x 16 elements, k = 2427 14.2 -> 12.8 us; 27 x 17, k = 636 5.4 -> 5.0.  In the kernels that hash between matrix instructions the
// merged form is the faster one (8192 x 768 -> 3072 random-bias shares: 3 %).
__device__ __forceinline__ uint32_t sq5_xor(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_xor_b32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ uint32_t sq5_tail_apart(uint32_t b)
{
    b = sq5_xor(b, b >> 9);
    b += SQ5_N2;
    b ^= (b >> 11);
    b *= SQ5_N3;
    b = sq5_xor(b, b >> 13);
    b += SQ5_N4;
    b ^= (b >> 15);
    b *= SQ5_N5;
    return b ^ (b >> 17);
}

// The same, four values at a time and written out, for kernels that do nothing but hash.  Two waves of a SIMD can have a vector instruction issued in
// the same four clocks, but only two of the simple kind (shift, exclusive or, addition: 2.05 clocks each then).  A product, a conversion, a matrix
// instruction, v_xad_u32 go alone, and the older wave goes first: while it has a vector instruction in every slot, the younger one stands at
// its first product until the older has left the loop, and nothing is issued together (54 clocks a hash for its 14 instructions, with 8, 4 and 2 waves a
// SIMD alike).  So those that go alone come in groups, and a wave at a group has the higher priority: the other one loses the slots of the group and no more.
// A hash, its conversion and its multiply-add: 56 -> 42 clocks, waits for LDS included.  (An s_nop on either side of every such instruction opens
// the slots too, 43 clocks, but only for waves in step: with LDS reads between 47 to 50.)
#define SQ5_SHIFTS(H, T, A, ADD, B)                                                                                      \
    "v_lshrrev_b32 " T ", " A ", " H "\n\tv_xor_b32 " H ", " T ", " H "\n\tv_add_u32 " H ", " ADD ", " H "\n\t"            \
    "v_lshrrev_b32 " T ", " B ", " H "\n\tv_xor_b32 " H ", " T ", " H "\n\t"
#define SQ5_FIRST(I0, I1, I2, I3) "s_setprio 1\n\t" I0 "\n\t" I1 "\n\t" I2 "\n\t" I3 "\n\ts_setprio 0\n\t"
#define SQ5_MUL(H, N) "v_mul_lo_u32 " H ", " H ", " N
// four values in place, from the first round's up to the last product; T a scratch register, N3 and N5 the multipliers
#define SQ5_FOUR(H0, H1, H2, H3, T, N3, N5)                                                                              \
    SQ5_SHIFTS(H0, T, "9", "0xa884f197", "11") SQ5_SHIFTS(H1, T, "9", "0xa884f197", "11")                                \
    SQ5_SHIFTS(H2, T, "9", "0xa884f197", "11") SQ5_SHIFTS(H3, T, "9", "0xa884f197", "11")                                \
    SQ5_FIRST(SQ5_MUL(H0, N3), SQ5_MUL(H1, N3), SQ5_MUL(H2, N3), SQ5_MUL(H3, N3))                                        \
    SQ5_SHIFTS(H0, T, "13", "0xb79f3abb", "15") SQ5_SHIFTS(H1, T, "13", "0xb79f3abb", "15")                              \
    SQ5_SHIFTS(H2, T, "13", "0xb79f3abb", "15") SQ5_SHIFTS(H3, T, "13", "0xb79f3abb", "15")                              \
    SQ5_FIRST(SQ5_MUL(H0, N5), SQ5_MUL(H1, N5), SQ5_MUL(H2, N5), SQ5_MUL(H3, N5))
static_assert(SQ5_N2 == 0xa884f197u && SQ5_N4 == 0xb79f3abbu, "the additions of SQ5_FOUR");

// sum += c[i] 2^31 noise(first + i N1), i = 0 .. 3, one fused multiply-add after the other; first += 4 N1
__device__ __forceinline__ void sq5_four_terms(uint32_t &first, float &sum, const float __attribute__((ext_vector_type(4))) &c)
{
    uint32_t h[4], t;
    asm("v_mov_b32 %0, %5\n\tv_add_u32 %1, 0xd2a80a3f, %5\n\tv_add_u32 %2, 0xa550147e, %5\n\tv_add_u32 %3, 0x77f81ebd, %5\n\t"
        SQ5_FOUR("%0", "%1", "%2", "%3", "%4", "%7", "%8")
        "v_lshrrev_b32 %4, 17, %0\n\tv_xor_b32 %0, %4, %0\n\tv_lshrrev_b32 %4, 17, %1\n\tv_xor_b32 %1, %4, %1\n\t"
        "v_lshrrev_b32 %4, 17, %2\n\tv_xor_b32 %2, %4, %2\n\tv_lshrrev_b32 %4, 17, %3\n\tv_xor_b32 %3, %4, %3\n\t"
        SQ5_FIRST("v_cvt_f32_i32 %0, %0", "v_cvt_f32_i32 %1, %1", "v_cvt_f32_i32 %2, %2", "v_cvt_f32_i32 %3, %3")
        "v_add_u32 %5, 0x4aa028fc, %5\n\t"
        "v_fmac_f32 %6, %0, %9\n\tv_fmac_f32 %6, %1, %10\n\tv_fmac_f32 %6, %2, %11\n\tv_fmac_f32 %6, %3, %12"
        : "=&v"(h[0]), "=&v"(h[1]), "=&v"(h[2]), "=&v"(h[3]), "=&v"(t), "+v"(first), "+v"(sum)
        : "s"(SQ5_N3), "s"(SQ5_N5), "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]));
}
static_assert(SQ5_N1 == 0xd2a80a3fu && 2u * SQ5_N1 == 0xa550147eu && 3u * SQ5_N1 == 0x77f81ebdu && 4u * SQ5_N1 == 0x4aa028fcu, "the additions of sq5_four_terms");

// h[i] = the hash of the first-round value f[i] + m, exclusive-or mask (in a vector register), for a matrix instruction that follows: it has the higher
// priority too, which the next call, or the kernel, takes back.  (The s_nop: two instructions have to lie between a vector instruction and a
// matrix instruction that reads its result.)
#define SQ5_MASKED(H, T, MASK) "v_lshrrev_b32 " T ", 17, " H "\n\tv_bitop3_b32 " H ", " T ", " H ", " MASK " bitop3:0x96\n\t"
__device__ __forceinline__ void sq5_eight_masked(const int __attribute__((ext_vector_type(4))) &f, const int __attribute__((ext_vector_type(4))) &g, uint32_t m,
                                                 uint32_t mask, int __attribute__((ext_vector_type(8))) &h)
{
    uint32_t t, v[8];
    asm("s_setprio 0\n\tv_add_u32 %0, %9, %17\n\tv_add_u32 %1, %10, %17\n\tv_add_u32 %2, %11, %17\n\tv_add_u32 %3, %12, %17\n\t"
        SQ5_FOUR("%0", "%1", "%2", "%3", "%8", "%19", "%20")
        SQ5_MASKED("%0", "%8", "%18") SQ5_MASKED("%1", "%8", "%18") SQ5_MASKED("%2", "%8", "%18") SQ5_MASKED("%3", "%8", "%18")
        "v_add_u32 %4, %13, %17\n\tv_add_u32 %5, %14, %17\n\tv_add_u32 %6, %15, %17\n\tv_add_u32 %7, %16, %17\n\t"
        SQ5_FOUR("%4", "%5", "%6", "%7", "%8", "%19", "%20")
        SQ5_MASKED("%4", "%8", "%18") SQ5_MASKED("%5", "%8", "%18") SQ5_MASKED("%6", "%8", "%18") SQ5_MASKED("%7", "%8", "%18")
        "s_setprio 1\n\ts_nop 0"
        : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]), "=&v"(t)
        : "v"(f[0]), "v"(f[1]), "v"(f[2]), "v"(f[3]), "v"(g[0]), "v"(g[1]), "v"(g[2]), "v"(g[3]), "v"(m), "v"(mask), "s"(SQ5_N3), "s"(SQ5_N5));
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = (int)v[i];
}

__device__ __forceinline__ uint32_t sq5_bits(uint32_t idx, uint32_t seed) { return sq5_tail(idx * SQ5_N1 + seed); }

// int32 reinterpretation -> fp32 (round to nearest even) -> exact scale by 2^-31
// (reference: RandumbTensor.py:162-163; fp32(1/0x7FFFFFFF) == 2^-31).
__device__ __forceinline__ float sq5_unit(uint32_t bits) { return (float)(int32_t)bits * 4.656612873077392578125e-10f; }

__device__ __forceinline__ float noise1d(uint32_t idx, uint32_t seed) { return sq5_unit(sq5_bits(idx, seed)); }
__device__ __forceinline__ float noise2d(uint32_t n, uint32_t m, uint32_t seed)
{
    return sq5_unit(sq5_bits(PRIME * n + m, seed));
}
// First-round value for (n, m): pass to sq5_tail.  first(n, m+1) = first(n, m) + N1; first(n+1, m) = first(n, m) + PN1.
__device__ __forceinline__ uint32_t sq5_first(uint32_t n, uint32_t m, uint32_t seed) { return n * PN1 + m * SQ5_N1 + seed; }

// ----------------------------------------------------------------------------------------------- bf16
typedef uint16_t bf16_t;  // storage type
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float bf16_to_f32(bf16_t h) { return __uint_as_float(((uint32_t)h) << 16); }
__device__ __forceinline__ uint32_t f32x2_to_bf16x2(float lo, float hi)
{
    f32x2 v = {lo, hi};
    bf16x2 r = __builtin_convertvector(v, bf16x2);  // v_cvt_pk_bf16_f32: round to nearest even
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ bf16_t f32_to_bf16(float f) { return (bf16_t)(f32x2_to_bf16x2(f, 0.0f) & 0xffffu); }
// two bf16 values in a word
__device__ __forceinline__ float lo_f32(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_f32(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ float relu(float v) { return v <= 0.0f ? 0.0f : v; }   // NaN stays NaN
__device__ __forceinline__ uint32_t relu2_pair(uint32_t w)
{
    const float a = relu(lo_f32(w)), b = relu(hi_f32(w));
    return f32x2_to_bf16x2(a * a, b * b);
}
// the gradient of relu(x)^2, d * 2 relu(x), of two values: 0 where x <= 0 whatever d is, an infinite or undefined one included
__device__ __forceinline__ uint32_t relu2_grad_pair(uint32_t x, uint32_t d)
{
    const float a = lo_f32(x), b = hi_f32(x);
    return f32x2_to_bf16x2(a <= 0.0f ? 0.0f : lo_f32(d) * (a + a), b <= 0.0f ? 0.0f : hi_f32(d) * (b + b));
}

template <typename T> struct elem;
template <> struct elem<float> {
    static constexpr int dtype = RDB_F32;
    __device__ static __forceinline__ float load(const float *p) { return *p; }
    __device__ static __forceinline__ void store(float *p, float v) { *p = v; }
    __device__ static __forceinline__ float round(float v) { return v; }
};
template <> struct elem<bf16_t> {
    static constexpr int dtype = RDB_BF16;
    __device__ static __forceinline__ float load(const bf16_t *p) { return bf16_to_f32(*p); }
    __device__ static __forceinline__ void store(bf16_t *p, float v) { *p = f32_to_bf16(v); }
    __device__ static __forceinline__ float round(float v) { return bf16_to_f32(f32_to_bf16(v)); }
};

// Reads element i of a buffer whose dtype is only known at run time.
__device__ __forceinline__ float load_as_f32(const void *p, int dtype, int64_t i)
{
    return dtype == RDB_BF16 ? bf16_to_f32(((const bf16_t *)p)[i]) : ((const float *)p)[i];
}

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ----------------------------------------------------------------------------------------------- timeline stamps
// RDB_STAMP(slot), slot 0..3, records when thread 0 of a block passes a point of a kernel.  Compiled out of the library.  A
// timing harness defines RDB_STAMPS and a __device__ pointer rdb_stamp_buf before including the kernel sources and then
// finds, per block, 4 kernels x 4 slots of two counters: the constant-rate wall clock (comparable across compute units) and
// the shader clock.  Which of the 4 kernels a launch is, the harness says with an expression RDB_STAMP_KERNEL_ID over the
// launch geometry (no extra registers or LDS in the kernels, so their occupancy is that of the library's build).
// 16-byte store of data that the kernel which writes it does not read again (it is for the next launch, on other dies):
// non-temporal, so the line does not wait dirty in this die's L2 for the write-back at the end of the kernel.
template <class V> __device__ __forceinline__ void store_stream(V *dst, const V &v)
{
#ifdef RDB_NO_STREAM_STORES
    *dst = v;
#else
    __builtin_nontemporal_store(v, dst);
#endif
}

// ----------------------------------------------------------------------------------------------- producer -> consumer blocks of one launch
// Blocks of one launch that consume what earlier blocks of the same launch produce: a producer publishes a 64-bit tag, unique
// to the launch, in a slot of its own when its output is in memory; a consumer polls the slots it depends on.  Hardware
// queues hand out the blocks of a launch in index order (per die), so a consumer that only waits for blocks with lower
// indices cannot starve them.  That order is what the hardware is seen to do, not something its documentation promises, so
// the wait is bounded: after `polls` polls (SYNC_SPIN_LIMIT: a fraction of a second) the consumer gives up.  A block that
// gives up never computes on what happens to be in memory: it counts itself in the library's per-device give-up counter
// (which the host reads: rdb_sync_giveups), sets bit 1 of *err when the caller has such a word, and its caller fills the
// block's share of the output with NaN and leaves.
//
// The dies' L2 caches are not coherent with each other, and the fences that make them so (write back / invalidate a whole
// L2) cost microseconds per block.  So the data that passes from producer to consumer goes around them instead: stored and
// loaded with device scope (SCOPE_DEVICE below: write-through, and read from memory), as the tags are.
constexpr int SYNC_SPIN_LIMIT = 1 << 17;
constexpr int SCOPE_DEVICE = 16;   // cache-policy argument of the raw buffer loads and stores: sc1

// What a waiting block needs besides its slots: how long to wait and where to report that it gave up.
struct SyncWait {
    unsigned int *err;       // NULL, or a word of the caller's state: bit 1 is set by a block that gave up
    unsigned int *giveups;   // the library's counter of such blocks on this device
    int polls;               // bound of the wait
};

// Device address of the give-up counter of the current device (rdb_error.hip); one per device, zero when the library loads.
int sync_giveups_ptr(unsigned int **out);
// The tag of a launch (never 0).
unsigned long long next_sync_tag();
// 1: the one-launch forms run where they apply; 0: producers and consumers always as separate launches (rdb_set_one_launch).
int one_launch_mode();

// All threads of the block call this after their last store (with SCOPE_DEVICE) of the block's output.
__device__ __forceinline__ void publish_tag(unsigned long long *slot, unsigned long long tag)
{
    __builtin_amdgcn_s_waitcnt(0);   // this wave's stores have been acknowledged at their scope
    __syncthreads();                 // ... and every other wave's
    if (threadIdx.x == 0) __hip_atomic_store(slot, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One wave calls this: lanes 0 .. n - 1 (n <= 64) poll slots[0 .. n - 1].  Returns false after the poll limit: the caller must
// then poison its output instead of computing it.  Loads of the producers' data that follow must use SCOPE_DEVICE.
__device__ __forceinline__ bool await_tags(const unsigned long long *slots, int n, unsigned long long tag, const SyncWait &w)
{
    const int lane = threadIdx.x & 63;
    const unsigned long long *mine = slots + (lane < n ? lane : 0);
    for (int it = 0; it < w.polls; ++it) {
        const unsigned long long v = __hip_atomic_load(mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__all(v == tag)) return true;
        __builtin_amdgcn_s_sleep(20);
    }
    if (lane == 0) {
        if (w.err) atomicOr(w.err, 2u);
        atomicAdd(w.giveups, 1u);
    }
    return false;
}

// Where a producer may still be on its way to memory that a consumer owns (sums on the way in its output's rows): a consumer that has
// given up leaves the launch's tag in a word of theirs before it poisons its output, and the producer looks at the word
// once its own stores are in memory.  Either the producer sees it and poisons what it wrote, or its stores came first.
__device__ __forceinline__ void mark_gone(unsigned int *word, unsigned long long tag)
{
    if ((threadIdx.x & 63) == 0) __hip_atomic_store(word, (unsigned int)tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);
}
__device__ __forceinline__ bool is_gone(const unsigned int *word, unsigned long long tag)
{
    return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned int)tag;
}

// The same wave calls this once its wait has succeeded.  A launch recorded in a graph runs again with the tag it was recorded
// with, so the slots must not still hold it then: every consumer of the n slots counts itself in `counter`, and the last of
// the `consumers` (all of them are past their wait by then) clears the slots.  The counter is set to zero by one of the
// producers of these slots before it publishes its tag (store it before the call of publish_tag).
__device__ __forceinline__ void release_tags(unsigned long long *slots, int n, unsigned int *counter, int consumers)
{
    const int lane = threadIdx.x & 63;
    unsigned int old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    old = (unsigned int)__builtin_amdgcn_readfirstlane((int)old);
    if (old == (unsigned int)(consumers - 1) && lane < n) __hip_atomic_store(slots + lane, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A sum over the blocks of a launch without a launch of its own: every block leaves its share and counts itself, and the last one adds the
// shares up, in an order that does not depend on who that is.  Counting one word costs 10 ns a block (1248 blocks: 13 us), so the blocks come in
// groups: the last of a group counts it.
struct BlockSum {
    float *part;             // one value per item
    unsigned int *arrived;   // a word for the groups, then one per group; zero when the launch begins (an earlier launch's business)
    void *out;
    int out_bf16;
};
// one thread of the block (always the same one)
__device__ __forceinline__ void leave_share(const BlockSum &q, int item, float v)
{
    __hip_atomic_store(q.part + item, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// all 256 threads of every block, after its last share, which thread 0 has left: block of `size` in `group` of `groups` (size 1: no words of their
// own); sh: 257 floats of LDS that nobody reads any more
__device__ __forceinline__ void sum_shares(const BlockSum &q, int items, int size, int group, int groups, float *sh)
{
    if (threadIdx.x == 0) {
        __builtin_amdgcn_s_waitcnt(0);   // the shares are in memory
        bool last = size == 1 || __hip_atomic_fetch_add(q.arrived + 1 + group, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned int)size - 1;
        if (last) last = __hip_atomic_fetch_add(q.arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned int)groups - 1;
        sh[256] = last ? 1.0f : 0.0f;
    }
    __syncthreads();
    if (sh[256] == 0.0f) return;
    float v = 0.0f;
    for (int i = threadIdx.x; i < items; i += 256) v += __hip_atomic_load(q.part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int h = 128; h >= 1; h >>= 1) {
        if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (q.out_bf16) *static_cast<bf16_t *>(q.out) = f32_to_bf16(sh[0]);
        else *static_cast<float *>(q.out) = sh[0];
    }
}

#ifdef RDB_STAMPS
#ifndef RDB_STAMP_KERNEL_ID
#define RDB_STAMP_KERNEL_ID 0
#endif
#define RDB_STAMP(slot)                                                                                                  \
    do {                                                                                                                 \
        if (threadIdx.x == 0 && rdb_stamp_buf) {                                                                         \
            const size_t at_ = ((size_t)blockIdx.x * 16 + (RDB_STAMP_KERNEL_ID) * 4 + (slot)) * 2;                       \
            rdb_stamp_buf[at_] = wall_clock64();                                                                         \
            rdb_stamp_buf[at_ + 1] = clock64();                                                                          \
        }                                                                                                                \
    } while (0)
#else
#define RDB_STAMP(slot) ((void)0)
#endif

}  // namespace rdb
