// Weight GEMM on the gfx950 matrix cores with the per-token epilogue in its
// store:
//
//   acc[t, n] = sum_k x[t, k] * w[n, k]        (f16 or bf16 operands, f32 sums)
//   out[t, n] = act(acc[t, n] + bias[n])        (t2h_linear)
//
// x is the token rows [rows, K] and w a linear's weight in its checkpoint
// layout [N, K]; both are K-contiguous, which is what the MFMA operands read.
// The weight rows are the MFMA's A operand and the token rows its B operand,
// so a 16x16x32 MFMA tile is 16 features x 16 tokens and each lane holds one
// token (lane % 16) and four consecutive features (4 * (lane / 16) + 0..3):
// a RoPE pair (2p, 2p + 1) stays in one lane.
//
// Products of two f16 (or bf16) values are exact in f32 and the sums are f32,
// as in the reference's 16-bit-weight kernel gemm_tiled_f16sh (both operands
// rounded to f16, f32 accumulation; gpu/linear.mojo:326-388, selected by
// GpuLinear.try_build 430-465); only the summation order differs.
//
// The main loop here (256 features x BT tokens, 8 waves) serves the large
// launches: MI355X runs them at its power limit (1.46-1.73 GHz over the four
// large products of a 201,436-token block instead of 2.4), so what counts is matrix-core work per joule and no idle matrix cores.
// - 16x16x32 MFMAs: a 256 x 256 tile of K = 6144 ran at 1,388 TFLOP/s with
//   them and at 1,160 with 32x32x16 in the same loop (f16, 201,436 tokens).
// - Direct-to-LDS loads (16 bytes per lane), no register staging.
// - Two groups of 4 waves (one of each per SIMD) take turns: while one runs 32
//   MFMAs (one 64-feature half of its wave tiles over 64 k) the other reads
//   its next fragments and issues the loads of two steps ahead; a barrier ends
//   each turn. 32 MFMAs a turn and not 16: 1,385 against 1,290 TFLOP/s. The
//   matrix cores are busy 70-72 % of a plain linear of K = 1536 (the two waves
//   per SIMD in step that this replaced: 66-67 %) and 76-78 % of K = 6144 with
//   the residual, epilogues included.
// - Persistent blocks: the next tile's first loads are issued before this
//   tile's epilogue (K = 1536: 1,284 -> 1,315 TFLOP/s).
// In all, at 201,436 tokens (f16, the former kernels and these in turn): K =
// 1536 to 6144 features 1,115 -> 1,253 TFLOP/s (hipBLASLt 1,257), with bias and
// GELU-tanh 1,022 -> 1,157-1,179; K = 6144 to 1536 features 1,212 -> 1,355
// (1,343), with the gated residual 1,167 -> 1,306.
//
// Reference: GpuLinear.enqueue_gemm (gpu/linear.mojo:535-560, c[m, co] =
// a[m, ci] @ W^T), the MLP's lin0 + gelu_tanh_bias (gpu/linear.mojo:662-684,
// 776-809).
#pragma once
#include "t2h_device.h"
#include "t2h_internal.h"
#include "t2h_act.h"
#include "t2h_rope.h"

namespace t2h {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;
template <> struct Mfma<_Float16> {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    __device__ static __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma<__bf16> {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    __device__ static __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};

constexpr int kBK = 64;                    // k per step: one 128-byte LDS row per operand row

// Slot of 16-byte k chunk c of LDS row r: c ^ swz(r). A fragment read takes
// chunk (4s + lane / 16) of rows lane % 16; the LDS serves a 16-byte read in
// four turns of 16 lanes (0-3, 12-15, 20-27 / 4-11, 16-19, 28-31 / the same
// + 32), and with this swizzle each turn's 16 chunks lie in distinct banks.
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

// Wait until at most N of this wave's vector-memory operations are pending
// (vmcnt only; gfx9 encoding: vmcnt[3:0] bits 3:0, vmcnt[5:4] bits 15:14).
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xC07F); }   // lgkmcnt(0)
// Block barrier that nothing is scheduled across.
__device__ __forceinline__ void turn_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// Tile u of a launch: token tile and feature tile. Tile numbers are dealt to
// the 8 XCDs in contiguous ranges (XCD x = blocks b with b % 8 == x) and run,
// within groups of tgroup token tiles, feature tile by feature tile, so the
// tiles resident on one XCD share a few weight and token slabs in its L2.
struct TileRange {
    int64_t lo, cnt;
    __device__ __forceinline__ TileRange(int64_t nb, int xcd) {
        const int64_t q = nb >> 3, r = nb & 7;
        lo = xcd * q + (xcd < r ? xcd : r);
        cnt = q + (xcd < r ? 1 : 0);
    }
};
__device__ __forceinline__ void tile_at(const GemmArgs& a, int64_t u, int64_t& tt, int64_t& ft) {
    const int64_t ntok = a.nblocks / a.ftiles;
    const int64_t gsz = (int64_t)a.tgroup * a.ftiles;
    const int64_t g = u / gsz, off = u - g * gsz;
    const int64_t rem = ntok - g * a.tgroup;
    const int64_t tg = rem < a.tgroup ? rem : a.tgroup;
    tt = g * a.tgroup + off % tg;
    ft = off / tg;
}
// Token tiles per group: 4, or 2 for K >= 4096, where a token tile's operand
// slab is 4 times as long (201,436 tokens, K = 6144: 2 and 4 within 0.7 %, 8
// is 3 % slower; K = 1536: 2, 4 and 8 within 1 %).
inline int tile_group(int k) { return k >= 4096 ? 2 : 4; }

// ---- 256 features x BT tokens, 8 waves --------------------------------------
constexpr int kBF = 256;          // features per tile
constexpr int kThreads = 512;
// Tile offsets within an operand are 32-bit: the launcher sends row strides
// above this many elements to the kernel with 64-bit ones.
constexpr int64_t kMaxStride32 = int64_t(1) << 22;

template <int BT> struct Big {
    static constexpr int kWT = BT / 4;              // tokens per wave
    static constexpr int kTJ = kWT / 16;            // 16-token MFMA tiles per wave (8 feature tiles)
    static constexpr int kStage = 32768 + BT * 128; // LDS bytes of one k step: A0, A1 (128 rows each), x
    static constexpr int kLX = BT / 64;             // loads per wave per step: x; A0 and A1 have 2 each
    static constexpr int kInFlight = 4 + kLX;       // loads of the two turns after one that is waited for
    static constexpr int kSpare = kStage + 16384;   // A1 of stage 1: free from a tile's last step until
                                                    // the first step of the next (16 KB)
    static_assert(BT % 64 == 0 && BT <= 256, "token tile");
};

// Swap the odd 16-lane rows of a with the even ones of b.
__device__ __forceinline__ void swap_rows16(float& a, float& b) {
    const auto w = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    a = __builtin_bit_cast(float, (uint32_t)w[0]);
    b = __builtin_bit_cast(float, (uint32_t)w[1]);
}

// (Not templates: hipcc's host pass drops a kernel template whose own body
// names these builtins with generic pointers, without an error before the link.)
__device__ __forceinline__ void load_lds16(const uint8_t* base, uint8_t* lds, int64_t off) {
    __builtin_amdgcn_global_load_lds(base + off, lds, 16, 0, 0);
}
// base + soff stays scalar: left to itself the compiler steps a 64-bit lane
// address per load through the k loop, 16 registers that it then spills.
// (A buffer load with the step as its scalar offset: 1-2 % slower.)
__device__ __forceinline__ void load_lds16(const uint8_t* base, uint32_t soff, uint32_t voff, uint8_t* lds) {
    uint64_t b = reinterpret_cast<uint64_t>(base) + soff;
    asm volatile("" : "+s"(b));
    __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint8_t*>(b) + voff, lds, 16, 0, 0);
}

// A wave's addresses in one tile. Feature half H's LDS row r holds weight row
// (r / 64) * 128 + H * 64 + r % 64, so that a wave's 128 features are
// consecutive; token rows are in order, those past the last read the last.
// A load's address is a scalar base (tile and k step) and a 32-bit lane
// offset; W64: 64-bit lane offsets, for row strides past kMaxStride32.
template <int BT, bool W64 = false> struct BigCtx {
    const uint8_t *w, *x;
    int64_t k2, ldx2;
    uint32_t vw, wk, vx[Big<BT>::kLX];      // W64: vx = the token rows
    uint8_t* lds;
    int fa, fb, wave, lane;
    __device__ __forceinline__ void init(const GemmArgs& a, uint8_t* lds_) {
        lds = lds_;
        lane = threadIdx.x & 63;
        wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
        const int fr = lane & 15, h = lane >> 4;
        fa = ((wave >> 2) * 64 + fr) * 128 + (h ^ swz(fr)) * 16;
        fb = ((wave & 3) * Big<BT>::kWT + fr) * 128 + (h ^ swz(fr)) * 16;
        k2 = (int64_t)a.k * 2;
        ldx2 = a.ldx * 2;
        wk = (uint32_t)k2;
        const int r0 = wave * 8 + lane / 8;
        vw = (uint32_t)r0 * wk + ((lane & 7) ^ swz(r0)) * 16;
    }
    __device__ __forceinline__ void tile(const GemmArgs& a, int64_t t0, int64_t n0) {
        w = static_cast<const uint8_t*>(a.w) + n0 * k2;
        x = static_cast<const uint8_t*>(a.x) + t0 * ldx2;
        const int last = (int)(a.rows - 1 - t0 < BT - 1 ? a.rows - 1 - t0 : BT - 1);
        const int r0 = wave * 8 + lane / 8;
#pragma unroll
        for (int i = 0; i < Big<BT>::kLX; ++i) {
            int t = i * 64 + r0;
            t = t < last ? t : last;
            vx[i] = W64 ? (uint32_t)t : (uint32_t)t * (uint32_t)ldx2 + ((lane & 7) ^ swz(r0)) * 16;
        }
    }
    template <int H> __device__ __forceinline__ void load_a(int ks) const {
        uint8_t* st = lds + (ks & 1) * Big<BT>::kStage + H * 16384 + wave * 1024;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if constexpr (W64) load_lds16(w + (int64_t)ks * (kBK * 2), st + i * 8192,
                                          (int64_t)(i * 128 + H * 64 + wave * 8 + lane / 8) * k2 + chunk());
            else load_lds16(w, (uint32_t)ks * (kBK * 2) + (uint32_t)(i * 128 + H * 64) * wk, vw, st + i * 8192);
        }
    }
    __device__ __forceinline__ void load_x(int ks) const {
        uint8_t* st = lds + (ks & 1) * Big<BT>::kStage + 32768 + wave * 1024;
#pragma unroll
        for (int i = 0; i < Big<BT>::kLX; ++i) {
            if constexpr (W64) load_lds16(x + (int64_t)ks * (kBK * 2), st + i * 8192, vx[i] * ldx2 + chunk());
            else load_lds16(x, (uint32_t)ks * (kBK * 2), vx[i], st + i * 8192);
        }
    }
    __device__ __forceinline__ int chunk() const { return ((lane & 7) ^ swz(wave * 8 + lane / 8)) * 16; }
    // The loads ahead of step 0: all of it, and A0 and x of step 1.
    __device__ __forceinline__ void prologue(int steps) const {
        load_x(0);
        load_a<0>(0);
        load_a<1>(0);
        if (steps > 1) {
            load_x(1);
            load_a<0>(1);
        }
    }
};

template <typename T, int BT, int H, bool W64>
__device__ __forceinline__ void read_a(typename Mfma<T>::v8 (&a)[2][4], const BigCtx<BT, W64>& c, int ks) {
    const uint8_t* st = c.lds + (ks & 1) * Big<BT>::kStage + H * 16384;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            a[s][i] = *reinterpret_cast<const typename Mfma<T>::v8*>(st + (c.fa ^ (s * 64)) + i * 2048);
}
template <typename T, int BT, bool W64>
__device__ __forceinline__ void read_b(typename Mfma<T>::v8 (&b)[2][Big<BT>::kTJ], const BigCtx<BT, W64>& c, int ks) {
    const uint8_t* st = c.lds + (ks & 1) * Big<BT>::kStage + 32768;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int j = 0; j < Big<BT>::kTJ; ++j)
            b[s][j] = *reinterpret_cast<const typename Mfma<T>::v8*>(st + (c.fb ^ (s * 64)) + j * 2048);
}
// One turn of the matrix cores: a feature half's tiles over one k step.
template <typename T, int BT, int H>
__device__ __forceinline__ void mma_turn(f32x4 (&acc)[8][Big<BT>::kTJ], const typename Mfma<T>::v8 (&a)[2][4],
                                         const typename Mfma<T>::v8 (&b)[2][Big<BT>::kTJ]) {
    wait_lds();          // the fragments are here; their LDS rows may be overwritten after the barrier
    turn_barrier();
    __builtin_amdgcn_s_setprio(1);
    // pairs of token tiles, so that two MFMAs in a row share the A operand (1 %)
#pragma unroll
    for (int jp = 0; jp < Big<BT>::kTJ; jp += 2)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = jp; j < jp + 2; ++j)
                    acc[H * 4 + i][j] = Mfma<T>::run(a[s][i], b[s][j], acc[H * 4 + i][j]);
    __builtin_amdgcn_s_setprio(0);
    turn_barrier();
}

// The tile's accumulators over all of k (the prologue's loads are in flight). Turns of step k, for each group of waves: [read x, A0 of k;
// load A1 of k + 1] MFMAs of half 0 [read A1 of k; load x, A0 of k + 2] MFMAs
// of half 1. Group 1 (waves 4-7) runs one turn behind group 0, so a barrier
// separates every read of a buffer from the loads that overwrite it (a turn
// waits for its own reads before its barrier), and a load is waited for two
// turns after its own. On return every wave has finished reading the stages.
template <typename T, int BT, bool W64>
__device__ __forceinline__ void big_mainloop(const BigCtx<BT, W64>& c, int steps, f32x4 (&acc)[8][Big<BT>::kTJ]) {
    using V8 = typename Mfma<T>::v8;
    constexpr int kTJ = Big<BT>::kTJ;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < kTJ; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (steps > 1) wait_vm<Big<BT>::kInFlight>();   // x, A0 of step 0: A1 of step 0 and step 1 stay in flight
    else wait_vm<0>();
    turn_barrier();
    V8 a[2][4], b[2][kTJ];
    if (c.wave >= 4) turn_barrier();
    for (int ks = 0; ks < steps; ++ks) {
        read_b<T, BT, W64>(b, c, ks);
        read_a<T, BT, 0, W64>(a, c, ks);
        if (ks + 1 < steps) {
            c.template load_a<1>(ks + 1);
            wait_vm<Big<BT>::kInFlight>();      // A1 of this step
        } else {
            wait_vm<0>();
        }
        mma_turn<T, BT, 0>(acc, a, b);
        read_a<T, BT, 1, W64>(a, c, ks);
        if (ks + 2 < steps) {
            c.load_x(ks + 2);
            c.template load_a<0>(ks + 2);
            wait_vm<Big<BT>::kInFlight>();      // x, A0 of the next step
        } else {
            wait_vm<0>();
        }
        mma_turn<T, BT, 1>(acc, a, b);
    }
    if (c.wave < 4) turn_barrier();
    turn_barrier();
}

// The lane number as a value of its own: what an epilogue derives from it is
// then not moved ahead of the tile loop, where it would sit in registers that
// the main loop needs (kept there, the fused qkv's addresses were spilled and
// reloaded in every k step: 2.5 times the time).
__device__ __forceinline__ int fresh_lane(int lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}

// A persistent block's tiles: its XCD's range, every (blocks per XCD)-th.
struct TileWalk {
    int64_t lo, cnt, i;
    int per;
    __device__ __forceinline__ explicit TileWalk(const GemmArgs& a) {
        const TileRange r(a.nblocks, (int)(blockIdx.x & 7));
        lo = r.lo;
        cnt = r.cnt;
        per = (int)(gridDim.x >> 3);
        i = blockIdx.x >> 3;
    }
    __device__ __forceinline__ bool more() const { return i < cnt; }
};
// Blocks of a persistent launch: one per CU, a multiple of the 8 XCDs, no more than needed.
inline dim3 persistent_grid(int64_t nblocks) {
    int64_t g = device_cu_count() / 8;
    if (g < 1) g = 1;
    const int64_t need = (nblocks + 7) / 8;
    return dim3((unsigned)(8 * (need < g ? need : g)));
}

// A 16-byte store of an epilogue whose wave instruction writes whole 128-byte
// lines: non-temporal, the GEMM never re-reads its outputs, so they need not
// displace operands in L2. (Non-temporal stores of half lines cost 5 %.)
__device__ __forceinline__ void out_store16(void* p, u32x4 w) {
    __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(p));
}
__device__ __forceinline__ void out_store16(float* p, f32x4 v) {
    __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(p));
}

template <int ACT>
__device__ __forceinline__ float epi_f(float acc, float b) {
    const float v = bias_add(acc, b);
    if constexpr (ACT < 0) return v;
    else return act_f<ACT>(v);
}

}  // namespace
}  // namespace t2h
