// Wide Cubic GEMM (prompt-sized M, bits <= 4) for gfx950:
// y[M,N] = x[M,K] . decode(W)[N,K]^T
//
// Same prepared weights and the same per-tile arithmetic as gemm_kernel: per
// (m-tile, tile, k-block, fragment) one v_mfma_f32_16x16x32 in the same order,
// every K partition of the plan summed from zero and the partitions added in
// ascending order, so a row's output is the same bits at every M >= 5 (and
// below where the small-row kernel, with partitions of its own, does not run).
//
// What bounds it: the matrix cores, if the rest hides under them.  gemm_kernel
// decodes each weight M / 128 times, feeds two MFMAs per A fragment read from
// LDS, and a split K writes and rereads M x N x split FP32 partials.  Here:
//  - A workgroup is eight waves over 256 rows x 128 columns, four waves down
//    and two across, a wave 64 x 64: each fragment read feeds four MFMAs.
//  - Wave w decodes column tile w of the k-block once for the workgroup and
//    hands the fragments over through LDS, 1 KB per (tile, fragment), each
//    lane writing and reading its own 16 bytes (no bank conflicts).
//  - Activations go straight to LDS (buffer_load ... lds), one k-block ahead,
//    two stages, in a slot order that serves both sides (slot_at).  With one
//    k-block of decoded fragments that fills the 160 KB.
//  - Two groups of four waves, one of each per SIMD, run half a fragment
//    apart: one reads while the other multiplies.  All eight waves in step
//    queue on the LDS together and then on the matrix cores together (down
//    projection below: 240 us in step, 200 apart).
//  - K partitions are folded in registers (`tot`), so K is never split over
//    workgroups and no FP32 partial reaches memory.
// Measured at M = 2048, W4 g128 (us, gemm_kernel -> this; a plain bf16 library
// product of the decoded matrix): 4096 -> 6144 161 -> 135 (89), 4096 -> 4096
// 107 -> 67 (57), 4096 -> 2 x 12288 463 -> 420 (279), 12288 -> 4096 268 -> 201
// (180).
// Time per k-block and round of 256 workgroups: 2.0 us, of which the MFMAs
// alone take 1.1; the DMA's and the LDS reads' latency inside the halves is
// the rest (without the DMA 1.8, without the code loads 1.9).
#include <type_traits>

#include "cubic_gemm_common.h"

namespace cubic {
namespace {
using namespace gemm;

typedef __attribute__((address_space(3))) void lds_void_t;

constexpr uint32_t kPastEnd = 0x80000000u;  // a buffer offset past every extent
constexpr int kWideWaves = 8, kWideThreads = kWideWaves * 64;
static_assert(kWideRows == 256 && kWideCols == kWideWaves * 16, "4 x 2 waves of 64 x 64");

// Slot of 16-byte chunk c of row r in its 256-byte LDS row.  The DMA fills
// slots in lane order, and the address coalescer takes four lanes at a time:
// four neighbouring slots hold the four chunks of one 64-byte segment (a
// scattered order reads 70 B/ns per CU, this one 93-100, a contiguous run
// 108).  A fragment read takes lanes (row r, chunk 4q + f) in groups of 16
// with two values of q; rotating the segments by -(r / 4) and the chunks in
// them by r spreads every group over all banks (590 B/ns per CU; the plain
// order c ^ r 304).
__device__ __forceinline__ int slot_at(int r, int c) { return ((c >> 2) ^ ((-(r >> 2)) & 3)) << 2 | ((c ^ r) & 3); }
__device__ __forceinline__ int chunk_at(int r, int slot) { return slot_at(r, slot); }  // its own inverse

// s_waitcnt vmcnt(n) lgkmcnt(0)
constexpr int wide_waits(int n) { return (n & 0xF) | (0x7 << 4) | ((n >> 4) << 14); }

template <int BITS, bool F16>
__global__ __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void wide_kernel(GemmArgs a) {
    static_assert(BITS <= 4, "level-table decode only");
    constexpr int W = BITS, MW = meta_words<BITS>();
    constexpr int MT = 4, R = kWideRows, C = kWideCols;
    constexpr int kAInstr = R / 32;  // DMA instructions per wave and k-block
    // two activation stages as LDS objects of their own: the compiler then
    // sees that a DMA into one cannot touch the reads of the other and does
    // not drain it for them
    __shared__ __attribute__((aligned(1024))) uint8_t as0[R * 256];
    __shared__ __attribute__((aligned(1024))) uint8_t as1[R * 256];
    __shared__ __attribute__((aligned(1024))) uint8_t bs[4][C * 64];  // [fragment][tile][lane]

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int q = lane >> 4, col = lane & 15;
    // waves w and w + 4 share a SIMD and are in different groups
    const int wm = wave & 3, wn = wave >> 2, group = wave >> 2;

    // Workgroup -> (row chunk, column block).  Workgroups go round robin over
    // the eight XCDs; XCD x takes the x-th eighth of the row-chunk major order,
    // so the workgroups of one XCD share row chunks (their activations stay in
    // that XCD's L2) and stream the columns past them.
    const int cols = a.wide_cols, total = cols * a.wide_chunks;
    int id = blockIdx.x;
    {
        const int per = total >> 3, rest = total & 7, xcd = id & 7;
        id = xcd * per + min(xcd, rest) + (id >> 3);
    }
    const int cb = id % cols, m0 = id / cols * R, n0 = cb * C;
    const int kb_end = a.k_blocks;

    // --- activation DMA ----------------------------------------------------
    // Instruction p of a wave fills 64 slots: its row 4 p + q, position col.
    // Each has a buffer of its own that ends with row M - 1: rows past M read
    // zero, and the 32-bit offsets span four rows only (ldx < 2^28: host).
    const int r0 = wave * kAInstr * 4;
    const int rows_left = min(R, a.m - m0) - r0;  // of the wave's rows
    const int64_t quad_stride = a.ldx * 4;        // elements
    const uint16_t* x_wave = a.x + (int64_t)(m0 + r0) * a.ldx;
    const uint32_t row_bytes = (uint32_t)(a.ldx * 2);
    const int whole_kbs = a.k / kKBlock;
    // row 4 p + q (r0 is a multiple of 32) has segment rotation -p and chunk
    // rotation q
    const uint32_t x_row = (uint32_t)q * row_bytes + 16u * ((col ^ q) & 3), x_seg = 64u * (col >> 2);
    auto dma = [&](int kb, uint8_t* stage, int p) {
        __attribute__((address_space(3))) uint8_t* xs =
            (__attribute__((address_space(3))) uint8_t*)(void*)stage + (wave * kAInstr + p) * 1024;
        const int left = min(rows_left - 4 * p, 4);
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(x_wave + p * quad_stride), 0,
            left <= 0 ? 0 : (int)((uint32_t)(left - 1) * row_bytes) + a.k * 2, 0x00020000);
        const uint32_t seg = x_seg ^ (64u * (-p & 3));
        uint32_t off = x_row + seg + (uint32_t)kb * 256u;
        if (kb >= whole_kbs) {  // chunks past K read as zero: an offset past the buffer's extent
            const int c = (int)(seg >> 4) + ((col ^ q) & 3);
            if (kb * kKBlock + 8 * c >= a.k) off = kPastEnd;
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void_t*)xs, 16, off, 0, 0, 0);
    };

    // --- codes and level tables of this wave's tile, two k-blocks ahead -------
    const int nt = min(cb * kWideWaves + wave, a.n_tiles - 1);
    const uint32_t* code_base = a.codes + (int64_t)nt * a.k_blocks * (kWave * W);
    const uint32_t* meta_base = a.meta + (int64_t)nt * a.groups_k * (16 * MW);
    const bool whole_groups = a.group_in % kKBlock == 0;
    // the group of the next k-block to load, and the k-blocks left in it
    // (whole-k-block groups: the loads walk K in order)
    const int gpk = whole_groups ? a.group_in / kKBlock : 1;
    int g_next = 0, g_left = gpk;
    uint32_t rc[2][W], rm[2][MW];
    auto load = [&](int kb, uint32_t (&c)[W], uint32_t (&mt)[MW]) {
        kb = min(kb, kb_end - 1);
        const int g = min(g_next, a.groups_k - 1);
        if (--g_left == 0) {
            g_left = gpk;
            ++g_next;
        }
        const __amdgpu_buffer_rsrc_t cr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint32_t*>(code_base + (int64_t)kb * (kWave * W)), 0, kWave * W * 4, 0x00020000);
        const int co = lane * W * 4;
        if constexpr (W == 1) {
            c[0] = __builtin_amdgcn_raw_buffer_load_b32(cr, co, 0, 2);  // nt
        } else if constexpr (W == 2) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(cr, co, 0, 2);
            c[0] = v[0]; c[1] = v[1];
        } else if constexpr (W == 3) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b96(cr, co, 0, 2);
            c[0] = v[0]; c[1] = v[1]; c[2] = v[2];
        } else {
            const u32x4_dev_t v = __builtin_amdgcn_raw_buffer_load_b128(cr, co, 0, 2);
            c[0] = v.x; c[1] = v.y; c[2] = v.z; c[3] = v.w;
        }
        // whole-k-block groups: one group's 16 columns; else a group per quarter
        int mo = col * (MW * 4), extent = 16 * MW * 4;
        const uint32_t* mb = meta_base + (int64_t)g * (16 * MW);
        if (!whole_groups) {
            const int gq = min((int)((uint32_t)(kb * 4 + q) / (uint32_t)(a.group_in >> 5)), a.groups_k - 1);
            mb = meta_base;
            mo += gq * (16 * MW * 4);
            extent = 0x7FFFFFFF;  // a tile's metadata is below 2^31 bytes: host
        }
        const __amdgpu_buffer_rsrc_t mr =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(mb), 0, extent, 0x00020000);
        if constexpr (MW == 4) {
            const u32x4_dev_t v = __builtin_amdgcn_raw_buffer_load_b128(mr, mo, 0, 0);
            mt[0] = v.x; mt[1] = v.y; mt[2] = v.z; mt[3] = v.w;
        } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(mr, mo, 0, 0);
            mt[0] = v[0]; mt[1] = v[1];
        }
    };
    uint4 d;  // the next fragment of the tile, decoded ahead of its hand-over
    auto decode = [&](const uint32_t (&c)[W], const uint32_t (&m)[MW], int f) {
        LevelTable lt;
        lt.lo_lo = m[0];
        lt.hi_lo = m[1];
        lt.lo_hi = MW == 4 ? m[MW == 4 ? 2 : 0] : 0u;
        lt.hi_hi = MW == 4 ? m[MW == 4 ? 3 : 1] : 0u;
        d = decode_fragment<BITS>(c, f, lt);
    };
    auto hand_over = [&](int f) { *reinterpret_cast<uint4*>(&bs[f][wave * 1024 + lane * 16]) = d; };

    floatx4_t acc[MT][4], tot[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
            tot[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        }

    // --- main loop --------------------------------------------------------------
    // Per fragment a wave runs a memory half (hand over a fragment decoded
    // before, read this one's operands, issue a part of the DMA) and a matrix
    // half (multiply, decode the next fragment).  Group 1 runs one half behind
    // group 0: in every interval between two barriers one group reads and the
    // other multiplies.  LDS reuse: fragment buffer f, read in f's memory
    // half (complete by the end of the matrix half after it), is rewritten in
    // the memory half two fragments later, two intervals before the next
    // k-block reads it; the activation stage that the DMA refills was last
    // read in the previous k-block's last memory half, which waits for its
    // reads before its barrier.
    constexpr int kPer = (kAInstr + 1) / 2;  // DMA instructions of memory halves 0 and 1
    // vector-memory operations younger than a k-block's DMA where it has to
    // have landed: the codes and table two k-blocks ahead
    constexpr int kInFlight = 2;
    // fragment f of row `col` of a 16-row block is chunk 4q + f: an XOR of the
    // address of fragment 0
    uint32_t a_addr = (uint32_t)(wm * MT * 4096 + col * 256 + slot_at(col, 4 * q) * 16);
    load(0, rc[0], rm[0]);
    load(1, rc[1], rm[1]);
#pragma unroll
    for (int p = 0; p < kAInstr; ++p) dma(0, as0, p);
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        decode(rc[0], rm[0], f);
        hand_over(f);
    }
    decode(rc[0], rm[0], 2);
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (group == 1) __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    int fold_at = a.blocks_per_split;
    auto step = [&](auto parity, int kb) {
        constexpr int P = decltype(parity)::value;  // of the k-block
        uint8_t* stage = P ? as1 : as0;
        uint8_t* next = P ? as0 : as1;
        const int kb1 = min(kb + 1, kb_end - 1);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            // memory half
            uint4 av[MT], bv[4];
            hand_over((f + 2) & 3);  // of this k-block, from f = 2 of the next
            asm volatile("" : "+v"(a_addr));  // not four addresses kept across the loop
#pragma unroll
            for (int i = 0; i < MT; ++i)
                av[i] = *reinterpret_cast<const uint4*>(stage + (a_addr ^ (uint32_t)(16 * f)) + i * 4096);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                bv[j] = *reinterpret_cast<const uint4*>(&bs[f][(wn * 4 + j) * 1024 + lane * 16]);
            __builtin_amdgcn_sched_barrier(0);
            if (f < 2) {
#pragma unroll
                for (int p = f * kPer; p < (f + 1) * kPer; ++p)
                    if (p < kAInstr) dma(kb1, next, p);
            }
            if (f == 0 && kb == fold_at) {  // a partition ended: add it, start the next from zero
                fold_at += a.blocks_per_split;
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        tot[i][j] += acc[i][j];
                        acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (f == 1) load(kb + 2, rc[P], rm[P]);
            __builtin_amdgcn_sched_barrier(0);
            if (f == 3) __builtin_amdgcn_s_waitcnt(wide_waits(kInFlight));  // next activations landed, reads done
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            // matrix half
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[i][j] = mfma16<F16>(av[i], bv[j], acc[i][j]);
            if (f == 0) decode(rc[P], rm[P], 3);
            else decode(rc[P ^ 1], rm[P ^ 1], f - 1);
            // the decode between the MFMAs, not after them
#pragma unroll
            for (int z = 0; z < 2 * MT; ++z) {
                __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);  // MFMA
                __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);  // VALU
            }
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int kb = 0;
    for (; kb + 1 < kb_end; kb += 2) {
        step(std::integral_constant<int, 0>{}, kb);
        step(std::integral_constant<int, 1>{}, kb + 1);
    }
    if (kb < kb_end) step(std::integral_constant<int, 0>{}, kb);
    if (group == 0) __builtin_amdgcn_s_barrier();  // pairs with group 1's first

    // --- epilogue -----------------------------------------------------------------
    __builtin_amdgcn_s_waitcnt(0);  // the last DMA (a repeat) has landed before LDS is reused
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) tot[i][j] += acc[i][j];
    // 16 rows x 64 columns at a time through a wave-private run of LDS (row
    // pitch 72), then 16-byte row segments
    uint16_t* out = reinterpret_cast<uint16_t*>(as0) + wave * 16 * 72;
    const int row0 = m0 + wm * 16 * MT, n = n0 + wn * 64 + (lane & 7) * 8;
    // the lane's eight columns: one member and 16-byte aligned rows, or one by one
    const int member = n < a.n ? n / a.n_member : 0, nl = n - member * a.n_member;
    uint16_t* y0 = member_row(a, member, 0) + nl;
    const int64_t ldy = member_ldy(a, member);
    const bool vec = n + 8 <= a.n && nl + 8 <= a.n_member &&
                     ((reinterpret_cast<uintptr_t>(y0) | (uintptr_t)ldy * 2) & 15) == 0;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[(4 * q + r) * 72 + j * 16 + col] = out_bits<F16>(tot[i][j][r]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = h * 8 + (lane >> 3), m = row0 + i * 16 + r;
            const uint4 v = *reinterpret_cast<const uint4*>(&out[r * 72 + (lane & 7) * 8]);
            if (m < a.m && vec) {
                *reinterpret_cast<uint4*>(y0 + (int64_t)m * ldy) = v;
            } else if (m < a.m) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int ne = n + e;
                    if (ne < a.n) {
                        const int me = ne / a.n_member;
                        const uint32_t word = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
                        member_row(a, me, m)[ne - me * a.n_member] = (uint16_t)(word >> (16 * (e & 1)));
                    }
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

template <int BITS>
hipError_t launch_wide_bits(const GemmArgs& a, hipStream_t s) {
    const dim3 grid(a.wide_cols * a.wide_chunks);
    if (a.f16) wide_kernel<BITS, true><<<grid, kWideThreads, 0, s>>>(a);
    else wide_kernel<BITS, false><<<grid, kWideThreads, 0, s>>>(a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_wide_gemm(const GemmArgs& a, hipStream_t s) {
    switch (a.bits) {
        case 1: return launch_wide_bits<1>(a, s);
        case 2: return launch_wide_bits<2>(a, s);
        case 3: return launch_wide_bits<3>(a, s);
        case 4: return launch_wide_bits<4>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace cubic
