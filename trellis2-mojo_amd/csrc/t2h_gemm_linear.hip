// The weight GEMM's linear and gated-residual kernels and their launchers:
// t2h_linear (out = act(acc + bias)) and t2h_linear_gate_residual (out = res +
// fl(fl(acc + bias) * gate[b(t)])). Large launches run on the persistent
// 256 x 256 main loop of t2h_gemm_core.h; launches whose 256 x 256 tiles
// would leave CUs idle, and row strides past its 32-bit offsets, on smaller
// tiles.
//
// Reference: GpuLinear.enqueue_gemm (gpu/linear.mojo:535-560), the MLP's
// lin0 + gelu_tanh_bias (gpu/linear.mojo:662-684, 776-809), the out-linears
// + gate_add_bias_rows (gpu/block.mojo:86-110, 317-397).
#include "t2h_gemm_core.h"

#include <type_traits>

namespace t2h {
namespace {

// The rounding sequence of the gated-residual kernel with h = the f32 sums.
__device__ __forceinline__ float join_f(float acc, bool has_bias, float b, bool has_gate, float g, float r) {
    float v = has_bias ? add_rn(acc, b) : acc;
    if (has_gate) v = mul_rn(v, g);
    return add_rn(r, v);
}

// The batch row of tokens [t0, t0 + n) when they share one, else -1.
__device__ __forceinline__ int64_t tile_batch(const BatchMap& bm, int64_t t0, int64_t n, int64_t rows) {
    const int64_t t1 = t0 + n < rows ? t0 + n - 1 : rows - 1;
    const int32_t b0 = bm.batch_of(t0);
    return bm.batch_of(t1) == b0 ? b0 : -1;
}

// ---- large launches: 256 x BT tiles, persistent -------------------------------
// LDS past the two stages: 4 KB per wave, through which 16 tokens x 256 bytes
// at a time turn from the MFMA layout into whole rows (chunk c of row r at
// c ^ r: conflict-free both ways).
constexpr int kRegion = 4096;

// bias (and the tile's gate row) in LDS: one float of each per thread 0-255,
// read from memory before the main loop.
struct TileParams {
    float b, g;
    __device__ __forceinline__ void fetch(const GemmArgs& a, int64_t n0, int64_t tile_b) {
        const int i = threadIdx.x & 255;
        b = a.bias != nullptr ? a.bias[n0 + i] : 0.0f;
        g = a.gate != nullptr && tile_b >= 0 ? a.gate[tile_b * a.gate_stride + n0 + i] : 0.0f;
    }
    __device__ __forceinline__ void stage(float* p) const {
        const int i = threadIdx.x & 255;
        if (threadIdx.x < 256) p[i] = b;
        else p[256 + i] = g;
        wait_lds();
        turn_barrier();
    }
};

// out = act(acc + bias): activation in the MFMA layout, one rounding to the
// output type. 16-bit: a wave's 16 tokens x 128 features per pass; f32: x 64.
template <typename T, typename O, int ACT, int BT>
__global__ __launch_bounds__(kThreads, 1) void gemm_kernel(GemmArgs a) {
    constexpr int kTJ = Big<BT>::kTJ;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * Big<BT>::kStage + 8 * kRegion];
    TileWalk walk(a);
    if (!walk.more()) return;
    BigCtx<BT> c;
    c.init(a, lds);
    const int steps = a.k / kBK;
    const int wf = c.wave >> 2, wt = c.wave & 3;
    uint8_t* region = lds + 2 * Big<BT>::kStage + c.wave * kRegion;
    const float* prm = reinterpret_cast<const float*>(lds + Big<BT>::kSpare) + wf * 128;
    O* __restrict__ out = static_cast<O*>(a.out);
    int64_t tt, ft;
    tile_at(a, walk.lo + walk.i, tt, ft);
    c.tile(a, tt * BT, ft * kBF);
    TileParams tp;
    tp.fetch(a, ft * kBF, -1);
    c.prologue(steps);
    while (true) {
        const int64_t t0 = tt * BT, n0 = ft * kBF;
        f32x4 acc[8][kTJ];
        big_mainloop<T, BT, false>(c, steps, acc);
        const int lane = fresh_lane(c.lane);
        const int fr = lane & 15, h = lane >> 4;
        walk.i += walk.per;
        const bool more = walk.more();
        const TileParams mine = tp;
        if (more) {
            tile_at(a, walk.lo + walk.i, tt, ft);
            c.tile(a, tt * BT, ft * kBF);
            tp.fetch(a, ft * kBF, -1);
            c.prologue(steps);
        }
        mine.stage(reinterpret_cast<float*>(lds + Big<BT>::kSpare));
        const int64_t tw = t0 + wt * Big<BT>::kWT, nw = n0 + wf * 128;
        f32x4 b4[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) b4[i] = *reinterpret_cast<const f32x4*>(prm + i * 16 + h * 4);
#pragma unroll
        for (int j = 0; j < kTJ; ++j) {
            if constexpr (sizeof(O) == 2) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = epi_f<ACT>(acc[i][j][e], b4[i][e]);
                    u32x2 w;
                    w.x = Word<O>::pack(v);
                    w.y = Word<O>::pack(v + 2);
                    *reinterpret_cast<u32x2*>(region + fr * 256 + (((i * 2 + (h >> 1)) ^ fr) * 16) + (h & 1) * 8) = w;
                }
                wait_lds();
#pragma unroll
                for (int it = 0; it < 4; ++it) {
                    const int r = it * 4 + h;
                    const u32x4 w = *reinterpret_cast<const u32x4*>(region + r * 256 + ((fr ^ r) * 16));
                    const int64_t t = tw + j * 16 + r;
                    if (t < a.rows) out_store16(out + t * a.ldo + nw + fr * 8, w);
                }
                wait_lds();
            } else {
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        f32x4 v;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = epi_f<ACT>(acc[hf * 4 + i][j][e], b4[hf * 4 + i][e]);
                        *reinterpret_cast<f32x4*>(region + fr * 256 + (((i * 4 + h) ^ fr) * 16)) = v;
                    }
                    wait_lds();
#pragma unroll
                    for (int it = 0; it < 4; ++it) {
                        const int r = it * 4 + h;
                        const f32x4 v = *reinterpret_cast<const f32x4*>(region + r * 256 + ((fr ^ r) * 16));
                        const int64_t t = tw + j * 16 + r;
                        if (t < a.rows) out_store16(reinterpret_cast<float*>(out) + t * a.ldo + nw + hf * 64 + fr * 4, v);
                    }
                    wait_lds();
                }
            }
        }
        if (!more) break;
    }
}

// out = res + fl(fl(acc + bias) * gate[b(t)]): the residual join of the block
// in the store of the GEMM that makes h, so h never reaches memory. The f32
// sums go through the wave's region, 16 tokens x 64 features at a time, so
// that residual and output move as whole 128-byte (16-bit) or 256-byte (f32)
// row pieces: half a wave tile's residual is requested before the next tile's
// operands, the other half while the first is joined. (Reading and writing
// the f32 residual in the MFMA layout, 32-byte pieces, the out projection of
// 39,804 tokens took 409-437 us; so 244-248.) out may alias res: every element is
// read before it is written, by the same thread.
template <typename T, typename O, int BT>
__global__ __launch_bounds__(kThreads, 1) void gemm_res_kernel(GemmArgs a) {
    constexpr int kTJ = Big<BT>::kTJ;
    constexpr int kE = 16 / (int)sizeof(O);       // features per 16-byte piece
    constexpr int kPR = 64 / kE;                  // lanes per row of a pass
    constexpr int kRI = 64 / kPR;                 // rows per instruction
    constexpr int kIt = 16 / kRI;                 // instructions per pass
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * Big<BT>::kStage + 8 * kRegion];
    TileWalk walk(a);
    if (!walk.more()) return;
    BigCtx<BT> c;
    c.init(a, lds);
    const int steps = a.k / kBK;
    const int wf = c.wave >> 2, wt = c.wave & 3;
    uint8_t* region = lds + 2 * Big<BT>::kStage + c.wave * kRegion;
    const float* prm = reinterpret_cast<const float*>(lds + Big<BT>::kSpare) + wf * 128;
    const BatchMap bm{a.batch.offsets, a.batch.rows_per_batch, a.batch.nbatch};
    const O* __restrict__ res = static_cast<const O*>(a.res);
    O* __restrict__ out = static_cast<O*>(a.out);
    const bool has_bias = a.bias != nullptr, has_gate = a.gate != nullptr;
    const int64_t last = a.rows - 1;
    // gate row of a tile when all its rows share one batch (block-uniform),
    // else -1: each token looks up its own
    int64_t tt, ft, next_b = 0;
    TileParams tp;
    auto begin = [&]() {
        tile_at(a, walk.lo + walk.i, tt, ft);
        c.tile(a, tt * BT, ft * kBF);
        if (has_gate) next_b = tile_batch(bm, tt * BT, BT, a.rows);
        tp.fetch(a, ft * kBF, next_b);
        c.prologue(steps);
    };
    begin();
    while (true) {
        const int64_t t0 = tt * BT, n0 = ft * kBF, tile_b = next_b;
        f32x4 acc[8][kTJ];
        big_mainloop<T, BT, false>(c, steps, acc);
        const int lane = fresh_lane(c.lane);
        const int fr = lane & 15, h = lane >> 4;
        const int pr = lane / kPR, pc = lane % kPR;
        const int64_t tw = t0 + wt * Big<BT>::kWT, nw = n0 + wf * 128 + pc * kE;
        u32x4 rv[kTJ][kIt];
        auto fetch = [&](int hf, int j) {
#pragma unroll
            for (int it = 0; it < kIt; ++it) {
                const int64_t t = tw + j * 16 + it * kRI + pr;
                rv[j][it] = __builtin_nontemporal_load(
                    reinterpret_cast<const u32x4*>(res + (t < last ? t : last) * a.ldo + nw + hf * 64));
            }
        };
#pragma unroll
        for (int j = 0; j < kTJ; ++j) fetch(0, j);
        __builtin_amdgcn_sched_barrier(0);
        walk.i += walk.per;
        const bool more = walk.more();
        const TileParams mine = tp;
        if (more) begin();
        mine.stage(reinterpret_cast<float*>(lds + Big<BT>::kSpare));
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int j = 0; j < kTJ; ++j) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    *reinterpret_cast<f32x4*>(region + fr * 256 + (((i * 4 + h) ^ fr) * 16)) = acc[hf * 4 + i][j];
                wait_lds();
                float b[kE], gt[kE];
#pragma unroll
                for (int q = 0; q < kE / 4; ++q) {
                    *reinterpret_cast<f32x4*>(b + q * 4) =
                        *reinterpret_cast<const f32x4*>(prm + hf * 64 + pc * kE + q * 4);
                    *reinterpret_cast<f32x4*>(gt + q * 4) =
                        *reinterpret_cast<const f32x4*>(prm + 256 + hf * 64 + pc * kE + q * 4);
                }
#pragma unroll
                for (int it = 0; it < kIt; ++it) {
                    const int r = it * kRI + pr;
                    const int64_t t = tw + j * 16 + r;
                    if (has_gate && tile_b < 0)
                        load_params<kE>(a.gate + bm.batch_of(t < last ? t : last) * a.gate_stride + nw + hf * 64, gt);
                    float v[kE], x[kE];
#pragma unroll
                    for (int q = 0; q < kE / 4; ++q)
                        *reinterpret_cast<f32x4*>(v + q * 4) = *reinterpret_cast<const f32x4*>(
                            region + r * 256 + (((pc * (kE / 4) + q) ^ r) * 16));
#pragma unroll
                    for (int q = 0; q < 4; ++q) Word<O>::unpack(rv[j][it][q], x + q * Word<O>::N);
#pragma unroll
                    for (int e = 0; e < kE; ++e) v[e] = join_f(v[e], has_bias, b[e], has_gate, gt[e], x[e]);
                    u32x4 w;
#pragma unroll
                    for (int q = 0; q < 4; ++q) w[q] = Word<O>::pack(v + q * Word<O>::N);
                    if (t < a.rows) out_store16(out + t * a.ldo + nw + hf * 64, w);
                }
                if (hf == 0) fetch(1, j);
                wait_lds();
            }
        if (!more) break;
    }
}

// ---- small launches: smaller tiles ---------------------------------------------
// BF features x BT tokens by WF x WT waves, for launches whose 256 x 256
// tiles would leave CUs idle; the point is to put a tile on every CU. NST
// stages of 32 * KK k are filled by direct-to-LDS loads up to NST - 1 stages
// ahead; a step's fragments are read while the previous step's MFMAs run, and
// one barrier per step both publishes a stage and frees one. What bounds it is
// the LDS (a small tile reuses little) and the latency of a step. us a launch,
// back to back on one set of operands (f16, bias), 256 x 256 tiles against
// these: 2,369 tokens, K = 6144 to 1536 features 95 -> 50 (228 tiles of 128 x
// 128 instead of 60; 62 as one launch of an MLP), K = 1536 to 1536 29.5 -> 17.7;
// 1,029 tokens, K = 1024 to 3072 22 -> 13.7; one token, K = 1536 to 9216, on 64
// x 64 7.6, on 256 x 128 21.
// The sums run over k in the main loop's order on every tile size, so a row's
// result depends neither on the row count nor on the kernel. (Splitting k over
// two or four groups of waves and adding through LDS was no faster.)
// W64: 64-bit operand offsets (row strides past kMaxStride32).
template <int BF, int BT, int WF, int WT, int KK, int NST> struct Small {
    static constexpr int kWaves = WF * WT;
    static constexpr int kSK = 32 * KK;                 // k per stage
    static constexpr int kNB = kSK / kBK;               // 64-k blocks per stage
    static constexpr int kFI = BF / WF / 16, kTJ = BT / WT / 16;
    static constexpr int kRG = (BF + BT) / 8;           // 1 KB row groups per 64-k block
    static constexpr int kBlock = (BF + BT) * 128, kStage = kBlock * kNB;
    static constexpr int kNL = kRG * kNB / kWaves;      // loads per wave and stage
    static_assert(kSK % kBK == 0 && kRG * kNB % kWaves == 0 && kFI % 2 == 0 && kTJ >= 1 && BF % 8 == 0, "layout");
    static_assert(NST * kStage <= 160 * 1024 && NST >= 2 && (NST - 1) * kNL < 64, "resources");
};

template <int ACT>
__device__ __forceinline__ void epi8(float (&f)[8], const float (&b)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = epi_f<ACT>(f[e], b[e]);
}

template <typename T, typename O, bool RES, bool W64, int BF, int BT, int WF, int WT, int KK, int NST>
__global__ __launch_bounds__(64 * WF * WT, 1) void gemm_small_kernel(GemmArgs a) {
    using S = Small<BF, BT, WF, WT, KK, NST>;
    using V8 = typename Mfma<T>::v8;
    using Off = typename std::conditional<W64, int64_t, uint32_t>::type;
    constexpr int kFI = S::kFI, kTJ = S::kTJ;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NST * S::kStage];
    const int64_t blk = block_linear();
    if (blk >= a.nblocks) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wf = wave / WT, wt = wave % WT;
    int64_t tt, ft;
    {
        const TileRange r(a.nblocks, (int)(blk & 7));
        tile_at(a, r.lo + (blk >> 3), tt, ft);
    }
    const int64_t t0 = tt * BT, n0 = ft * BF;
    const uint8_t* wb = static_cast<const uint8_t*>(a.w) + n0 * a.k * 2;
    const uint8_t* xb = static_cast<const uint8_t*>(a.x) + t0 * a.ldx * 2;
    const int lastt = (int)(a.rows - 1 - t0 < BT - 1 ? a.rows - 1 - t0 : BT - 1);
    const int nkb = a.k / kBK, nst = (nkb + S::kNB - 1) / S::kNB;
    // load j of a wave: 1 KB group L = j * waves + wave of the stage: 64-k block
    // L / kRG, operand rows 8 * (L % kRG) + lane / 8
    Off vo[S::kNL];
#pragma unroll
    for (int j = 0; j < S::kNL; ++j) {
        const int r = ((j * S::kWaves + wave) % S::kRG) * 8 + lane / 8;
        const int rt = r - BF < lastt ? r - BF : lastt;
        const Off row = r < BF ? (Off)r * (Off)a.k : (Off)rt * (Off)a.ldx;
        vo[j] = row * 2 + ((lane & 7) ^ swz(r)) * 16;
    }
    auto issue = [&](int s) {     // past the last 64-k block: that block again, never used
        uint8_t* st = lds + (s % NST) * S::kStage + wave * 1024;
#pragma unroll
        for (int j = 0; j < S::kNL; ++j) {
            const int L = j * S::kWaves + wave;
            int kb = s * S::kNB + L / S::kRG;
            kb = kb < nkb ? kb : nkb - 1;
            const uint8_t* base = (L % S::kRG) * 8 < BF ? wb : xb;
            load_lds16(base + (int64_t)kb * (kBK * 2), st + j * S::kWaves * 1024, (int64_t)vo[j]);
        }
    };
    const int fr = lane & 15, h = lane >> 4;
    const int fa = (wf * kFI * 16 + fr) * 128 + (h ^ swz(fr)) * 16;
    const int fb = (BF + wt * kTJ * 16 + fr) * 128 + (h ^ swz(fr)) * 16;
    auto frags = [&](V8 (&A)[KK][kFI], V8 (&B)[KK][kTJ], int s) {
        const uint8_t* st = lds + (s % NST) * S::kStage;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const int off = (kk >> 1) * S::kBlock, x = (kk & 1) * 64;
#pragma unroll
            for (int i = 0; i < kFI; ++i) A[kk][i] = *reinterpret_cast<const V8*>(st + off + (fa ^ x) + i * 2048);
#pragma unroll
            for (int j = 0; j < kTJ; ++j) B[kk][j] = *reinterpret_cast<const V8*>(st + off + (fb ^ x) + j * 2048);
        }
    };
    f32x4 acc[kFI][kTJ];
#pragma unroll
    for (int i = 0; i < kFI; ++i)
#pragma unroll
        for (int j = 0; j < kTJ; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // step s: its fragments are in A, B; stage s + 1 is waited for, and after
    // the barrier every wave has read stage s, whose buffer takes stage s + NST
    auto step = [&](V8 (&A)[KK][kFI], V8 (&B)[KK][kTJ], V8 (&An)[KK][kFI], V8 (&Bn)[KK][kTJ], int s) {
        wait_lds();
        wait_vm<(NST - 2) * S::kNL>();
        turn_barrier();
        issue(s + NST);
        frags(An, Bn, s + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
            if (kk < 2 || s * S::kNB + (kk >> 1) < nkb) {      // a last stage may be partly past k
#pragma unroll
                for (int i = 0; i < kFI; ++i)
#pragma unroll
                    for (int j = 0; j < kTJ; ++j) acc[i][j] = Mfma<T>::run(A[kk][i], B[kk][j], acc[i][j]);
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    V8 af[2][KK][kFI], bf[2][KK][kTJ];
#pragma unroll
    for (int s = 0; s < NST; ++s) issue(s);
    wait_vm<(NST - 1) * S::kNL>();
    turn_barrier();
    frags(af[0], bf[0], 0);
    int s = 0;
    for (; s + 1 < nst; s += 2) {
        step(af[0], bf[0], af[1], bf[1], s);
        step(af[1], bf[1], af[0], bf[0], s + 1);
    }
    if (s < nst) step(af[0], bf[0], af[1], bf[1], s);
    // the loads issued past the last stage land in LDS that only this block
    // owns, and a wave's end waits for its outstanding memory operations

    const BatchMap bm{a.batch.offsets, a.batch.rows_per_batch, a.batch.nbatch};
    const bool has_bias = a.bias != nullptr, has_gate = RES && a.gate != nullptr;
    O* __restrict__ out = static_cast<O*>(a.out);
    const O* __restrict__ res = static_cast<const O*>(a.res);
#pragma unroll
    for (int i = 0; i < kFI; i += 2)
#pragma unroll
        for (int j = 0; j < kTJ; ++j) {
            // swapping 16-lane rows of two feature tiles gives each lane 8 consecutive
            // features of its token: tile i + (h & 1), features 8 * (h >> 1) + 0..7
            float f[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float p0 = acc[i][j][e], p1 = acc[i + 1][j][e];
                swap_rows16(p0, p1);
                f[e] = p0;
                f[4 + e] = p1;
            }
            const int64_t t = t0 + (wt * kTJ + j) * 16 + fr;
            const int64_t n = n0 + (wf * kFI + i + (h & 1)) * 16 + (h >> 1) * 8;
            if (t >= a.rows) continue;
            float b[8], gt[8], x[8];
            if (has_bias) {
                load_params<8>(a.bias + n, b);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) b[e] = 0.0f;
            }
            if constexpr (RES) {
                if (has_gate) load_params<8>(a.gate + bm.batch_of(t) * a.gate_stride + n, gt);
                load_elems<O, 8>(res + t * a.ldo + n, x);
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] = join_f(f[e], has_bias, b[e], has_gate, gt[e], x[e]);
            } else {
                switch (a.act) {      // uniform; one kernel for all activations
                    case T2H_ACT_RELU: epi8<T2H_ACT_RELU>(f, b); break;
                    case T2H_ACT_SILU: epi8<T2H_ACT_SILU>(f, b); break;
                    case T2H_ACT_GELU: epi8<T2H_ACT_GELU>(f, b); break;
                    case T2H_ACT_GELU_TANH: epi8<T2H_ACT_GELU_TANH>(f, b); break;
                    default: epi8<-1>(f, b); break;
                }
            }
            store_elems<O, 8>(out + t * a.ldo + n, f);
        }
}

template <typename T, typename O, bool RES, bool W64, int BF, int BT, int WF, int WT, int KK, int NST>
hipError_t launch_small(GemmArgs a, hipStream_t s) {
    a.ftiles = a.n / BF;
    a.nblocks = ((a.rows + BT - 1) / BT) * a.ftiles;
    hipLaunchKernelGGL((gemm_small_kernel<T, O, RES, W64, BF, BT, WF, WT, KK, NST>), grid_1d(a.nblocks),
                       dim3(64 * WF * WT), 0, s, a);
    return hipGetLastError();
}

// Tile choice: the least modelled time, rounds * (base + perk * K / 1024) us
// for rounds = ceil(tiles / CUs). The constants are least-squares readings of
// each tile timed over 1 to 20,000 rows, K 256 to 6,144 and N 1,024 to 9,216
// (f16, no epilogue): small tiles win while the larger ones leave CUs idle,
// large ones where all are busy, e.g. N = K = 1536: 32 x 64 to ~340 rows, 64 x
// 64 to ~680, 128 x 64 to ~1,360, 128 x 128 to ~2,700, 256 x 128 to ~5,400,
// then 256 x 256. It ranks the tiles and is no prediction: launches of one to
// three rounds, 1 to 39,804 rows at seven (N, K), measured 4 % below to 49 %
// above it (bias, GELU, f32 output; mean 22 %), to 70 % with a 16-bit residual
// and 137 % with an f32 one. The choice was the fastest tile within 0.3 %
// without a residual, within 8 % (0.2 % on average) with a 16-bit residual and
// within 21 % (1.5 %) with an f32 one, whose epilogue costs the large tiles more.
enum GemmPlan { kPlanBig, kPlan128, kPlan128x64, kPlan64, kPlan32x64, kPlanBig128, kPlanWide };
struct PlanCost {
    GemmPlan plan;
    int bf, bt;
    float base, perk;
};
constexpr PlanCost kPlanCosts[] = {
    {kPlan32x64, 32, 64, 2.2f, 2.1f},   {kPlan64, 64, 64, 2.6f, 2.9f},        {kPlan128x64, 128, 64, 2.7f, 5.0f},
    {kPlan128, 128, 128, 3.2f, 7.3f},   {kPlanBig128, 256, 128, 5.0f, 11.0f}, {kPlanBig, 256, 256, 8.0f, 15.5f},
};
GemmPlan gemm_plan(const GemmArgs& a) {
    if (a.ldx > kMaxStride32 || a.k > kMaxStride32) return kPlanWide;
    const int64_t cus = device_cu_count();
    GemmPlan best = kPlanBig;
    float least = 0.0f;
    for (const PlanCost& c : kPlanCosts) {
        const int64_t tiles = ((a.rows + c.bt - 1) / c.bt) * (a.n / c.bf);
        const float cost = (float)((tiles + cus - 1) / cus) * (c.base + c.perk * (float)a.k / 1024.0f);
        if (least == 0.0f || cost <= least) {
            least = cost;
            best = c.plan;
        }
    }
    return best;
}

template <typename T, typename O, bool RES>
hipError_t gemm_small(const GemmArgs& a, GemmPlan plan, hipStream_t s) {
    switch (plan) {
        case kPlan128: return launch_small<T, O, RES, false, 128, 128, 2, 4, 2, 4>(a, s);
        case kPlan128x64: return launch_small<T, O, RES, false, 128, 64, 4, 2, 2, 6>(a, s);
        case kPlan64: return launch_small<T, O, RES, false, 64, 64, 2, 4, 4, 4>(a, s);
        case kPlan32x64: return launch_small<T, O, RES, false, 32, 64, 1, 4, 4, 4>(a, s);
        default: return launch_small<T, O, RES, true, 64, 64, 2, 4, 4, 4>(a, s);
    }
}

template <typename T, typename O, int ACT, bool RES, int BT>
hipError_t launch_big(GemmArgs a, hipStream_t s) {
    a.ftiles = a.n / kBF;
    a.nblocks = ((a.rows + BT - 1) / BT) * a.ftiles;
    const dim3 g = persistent_grid(a.nblocks);
    if constexpr (RES) hipLaunchKernelGGL((gemm_res_kernel<T, O, BT>), g, dim3(kThreads), 0, s, a);
    else hipLaunchKernelGGL((gemm_kernel<T, O, ACT, BT>), g, dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

template <typename T, typename O, int ACT, bool RES>
hipError_t gemm_run(GemmArgs a, hipStream_t s) {
    a.tgroup = tile_group(a.k);
    const GemmPlan plan = gemm_plan(a);
    if (plan == kPlanBig) return launch_big<T, O, ACT, RES, 256>(a, s);
    if (plan == kPlanBig128) return launch_big<T, O, ACT, RES, 128>(a, s);
    return gemm_small<T, O, RES>(a, plan, s);
}

template <typename T, typename O>
hipError_t gemm_act(const GemmArgs& a, hipStream_t s) {
    switch (a.act) {
        case T2H_ACT_RELU: return gemm_run<T, O, T2H_ACT_RELU, false>(a, s);
        case T2H_ACT_SILU: return gemm_run<T, O, T2H_ACT_SILU, false>(a, s);
        case T2H_ACT_GELU: return gemm_run<T, O, T2H_ACT_GELU, false>(a, s);
        case T2H_ACT_GELU_TANH: return gemm_run<T, O, T2H_ACT_GELU_TANH, false>(a, s);
        default: return gemm_run<T, O, -1, false>(a, s);
    }
}

template <typename T>
hipError_t gemm_typed(const GemmArgs& a, hipStream_t s) {
    if (a.out_dtype == T2H_F32) return gemm_act<T, float>(a, s);
    return gemm_act<T, T>(a, s);
}

template <typename T>
hipError_t gemm_res_typed(const GemmArgs& a, hipStream_t s) {
    if (a.out_dtype == T2H_F32) return gemm_run<T, float, -1, true>(a, s);
    return gemm_run<T, T, -1, true>(a, s);
}

}  // namespace

int32_t gemm_feature_tile() { return kBF; }
int32_t gemm_k_step() { return kBK; }

hipError_t launch_gemm(GemmArgs a, hipStream_t s) {
    if (a.rows == 0) return hipSuccess;
    if (a.dtype == T2H_F16) return gemm_typed<_Float16>(a, s);
    return gemm_typed<__bf16>(a, s);
}

hipError_t launch_gemm_residual(GemmArgs a, hipStream_t s) {
    if (a.rows == 0) return hipSuccess;
    if (a.dtype == T2H_F16) return gemm_res_typed<_Float16>(a, s);
    return gemm_res_typed<__bf16>(a, s);
}

}  // namespace t2h
