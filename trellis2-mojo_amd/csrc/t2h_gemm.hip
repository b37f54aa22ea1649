// The qkv linear fused with the self-attention epilogue and the head-major
// pack (t2h_qkv_linear_pack), on the persistent main loop of t2h_gemm_core.h:
// a wave's 128 features are one head of 128 or two heads of 64.
//
// Reference: the qkv enqueue_gemm + bias_rms_rope_qkv + pack_q_z + pack_kv_z
// of the self-attention chain (gpu/attention.mojo:507-563, 566-594, 634-662,
// sequence 983-1013).
#include "t2h_gemm_core.h"

namespace t2h {
namespace {

// ---- qkv linear + attention epilogue + head-major pack ----------------------
// The qkv GEMM's output [rows, 3, H, HD] never reaches memory. A tile's 256
// features lie in one of q, k and v (H * HD is a multiple of 256). Per token,
// in the order of the separate kernels (bias_rms_rope_qkv, pack_q_z,
// pack_kv_z): + bias; q/k: RMS over the head, x * rsqrt(sum x^2) * (gamma *
// sqrt(D)); q/k: RoPE on the in-lane pairs (2p, 2p + 1) with cos/sin from the
// phase table or from the token's position; q: * 1/sqrt(D); tokens >= rows: 0.
// A token's head lies in the four lanes l, l ^ 16, l ^ 32, l ^ 48.
//
// cos/sin from positions: computing them per head and token (64 sincosf per
// token and head) took 395 us of the 3,243 us of 201,436 tokens x 4608
// features. Voxel coordinates are small integers, so each block computes
// cos/sin of every (position, frequency) once, into LDS, with the same sincosf
// of the same f32 angle, and its tiles look them up: the first 167 positions
// for 21 frequencies (heads of 128, three axes), 256 for 10 (heads of 64). 16
// tokens of which one lies outside are computed, from the positions and
// frequencies in LDS. us, all inside / all outside / no table (f16, bias, RMS):
// heads of 128, 2,369 tokens 48 / 56 / 61, 39,804 529 / 590 / 654, 201,436
// 2,690 / 2,930 / 3,250; heads of 64, 39,804 255 / 275 / 344.
//
// The values leave as whole 128-byte row pieces: through 2 KB of LDS per wave
// (16 tokens x 64 features) for qh [H, mp, D], k [H, lp, D], vh [H, lp, D];
// for the transposed k [H, D, lp] through the wave's share of the two stages,
// where 8 tokens of one feature are gathered per lane (such a tile requests
// the next tile's operands only afterwards). Tiles past the last token row
// skip the GEMM and write the pads.
constexpr int kHead = 128;                     // features of a wave
constexpr int kPos = 256;                      // most positions of the cos/sin table
// LDS past the stages: [wave half][bias, gamma * sqrt(D)][128] f32, the slots'
// table columns and frequencies, the tile's positions ([axes 0, 2 | axes 1,
// 3][256], two 16-bit halves a word), the table
constexpr int kSlotOff = 2048, kFreqOff = kSlotOff + 256, kPosOff = kFreqOff + 256, kExtra = 32768;
static_assert(T2H_MAX_POS_DIM == 4, "two words of two axes");
constexpr int kFar = -32768;                   // lower half: a coordinate past 16 bits, read again where needed

// Slot of a 16-byte chunk in a staged 256-byte token row: chunk c of row r
// at c ^ stage_swz(r). Over 16 consecutive rows (one write) every slot appears
// once; over rows 8g + j, g = 0..7 (one transposed gather) the slots are
// distinct; a row's 16 chunks are a permutation.
__device__ __forceinline__ int stage_swz(int r) { return ((r >> 3) ^ ((r & 7) << 1)) & 15; }

typedef float f32x16 __attribute__((ext_vector_type(16)));

// A launch parameter as a value of its own: a divisor's reciprocal or a flag
// derived from it would be computed ahead of the tile loop and sit, or be
// spilled, in registers that the loop needs.
template <typename V> __device__ __forceinline__ V fresh(V d) {
    asm volatile("" : "+s"(d));
    return d;
}

template <typename T, bool KT, int HD, int BT, bool W64>
__global__ __launch_bounds__(kThreads, 1) void qkv_pack_kernel(GemmArgs g, PackArgs p, RopeSlots tab) {
    constexpr int kTJ = Big<BT>::kTJ;
    constexpr int NH = kHead / HD;    // heads per wave
    constexpr int FPH = 8 / NH;       // 16-feature MFMA tiles per head
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * Big<BT>::kStage + kExtra];
    TileWalk walk(g);
    if (!walk.more()) return;
    BigCtx<BT, W64> c;
    c.init(g, lds);
    const int steps = g.k / kBK;
    const int wave = c.wave;
    const int wf = wave >> 2, wt = wave & 3;
    uint8_t* extra = lds + 2 * Big<BT>::kStage;
    const float* pb = reinterpret_cast<const float*>(extra) + (wf * 2 + 0) * kHead;
    const float* pg = reinterpret_cast<const float*>(extra) + (wf * 2 + 1) * kHead;
    const bool lookup = p.use_rope && p.phases == nullptr && g.rows > 0;
    const int fd = p.freq_dim;
    const int tab_off = kPosOff + (p.pos_dim > 1 ? 2048 : 1024);
    const int fit = fd > 0 ? ((kExtra - tab_off) / 8 - 1) / fd : 0;
    const int npos = fit < kPos ? fit : kPos;

    int64_t tt, ft;
    tile_at(g, walk.lo + walk.i, tt, ft);
    if (tt * BT < g.rows) {
        c.tile(g, tt * BT, ft * kBF);
        c.prologue(steps);
    }
    if (lookup) {
        // entry pos * fd + f: (cos, sin); the last entry is the identity. A
        // slot's word: its column's byte offset | axis << 16 (4: none)
        const float* freqs = reinterpret_cast<const float*>(extra + kFreqOff);
        float2* t = reinterpret_cast<float2*>(extra + tab_off);
        if (threadIdx.x < HD / 2) {
            const int ax = slot_axis(threadIdx.x, fd, p.pos_dim);
            reinterpret_cast<uint32_t*>(extra + kSlotOff)[threadIdx.x] =
                ax < 0 ? (uint32_t)(npos * fd * 8) | (4u << 16) : (uint32_t)((threadIdx.x - ax * fd) * 8) | (ax << 16);
            reinterpret_cast<float*>(extra + kFreqOff)[threadIdx.x] = tab.freq[threadIdx.x];
        }
        if (threadIdx.x == 0) t[npos * fd] = float2{1.0f, 0.0f};
        wait_lds();
        turn_barrier();
        if (fd > 0) {
            int pos = threadIdx.x / fd, f = threadIdx.x - pos * fd;
            const int dp = kThreads / fd, df = kThreads - dp * fd;
            while (pos < npos) {
                const float x = (float)pos;
                float cv, sv;
                slot_phase(&x, 0, freqs[f], cv, sv);
                t[pos * fd + f] = float2{cv, sv};
                pos += dp + (f + df >= fd);
                f += df - (f + df >= fd ? fd : 0);
            }
        }
        wait_lds();
    }
    while (true) {
        const int64_t t0 = tt * BT, n0 = ft * kBF;
        const int hg = (int)(n0 / HD);
        const int which = hg / p.heads;          // 0 q, 1 k, 2 v
        const int z = hg - which * p.heads + wf * NH;      // the wave's first head
        const float* __restrict__ bias = which == 0 ? p.bias_q : which == 1 ? p.bias_k : p.bias_v;
        const float* __restrict__ gamma = which == 0 ? p.gamma_q : which == 1 ? p.gamma_k : nullptr;
        const bool rope = p.use_rope && which < 2 && g.rows > 0;
        // one bias or gamma value and one word of positions per thread, read
        // ahead of the main loop and staged in LDS after it
        float pv;
        {
            const int i = threadIdx.x, f = (hg - which * p.heads) * HD + (i >> 8) * kHead + (i & 127);
            const float* src = (i >> 7) & 1 ? gamma : bias;
            pv = src != nullptr ? src[f] : 0.0f;
            if ((i >> 7) & 1) pv *= p.rms_scale;
        }
        const int pax = wave / (BT / 64);       // axes pax and pax + 2, or (0) the phase table's row
        const bool has_pos = rope && pax < (lookup ? p.pos_dim < 2 ? 1 : 2 : 1);
        uint32_t pw = 0;
        if (has_pos) {
            const int64_t t = t0 + threadIdx.x % BT, tc = t < g.rows ? t : g.rows - 1;
            if (!lookup) {
                pw = (uint32_t)(tc % fresh(p.phase_rows));
            } else {
                const PosSource src{fresh(p.coords), p.coord_cols, fresh(p.grid_res), p.pos_dim};
                const int lo = src.at(tc, pax), hi = pax + 2 < fresh(p.pos_dim) ? src.at(tc, pax + 2) : 0;
                const bool near = lo == (int16_t)lo && hi == (int16_t)hi && lo != kFar;
                pw = near ? (uint32_t)(uint16_t)lo | (uint32_t)hi << 16 : (uint32_t)(uint16_t)kFar;
            }
        }
        f32x4 acc[8][kTJ];
        if (t0 < g.rows) {
            big_mainloop<T, BT, W64>(c, steps, acc);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int j = 0; j < kTJ; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            turn_barrier();      // the last tile's LDS is read
        }
        const int lane = fresh_lane(c.lane);
        const int fr = lane & 15, h = lane >> 4;
        walk.i += walk.per;
        const bool more = walk.more();
        if (more) tile_at(g, walk.lo + walk.i, tt, ft);
        const bool next = more && tt * BT < g.rows;
        const bool trans = KT && which == 1;
        if (next) {
            c.tile(g, tt * BT, ft * kBF);
            if (!trans) c.prologue(steps);
        }
        reinterpret_cast<float*>(extra)[threadIdx.x] = pv;
        if (has_pos) reinterpret_cast<uint32_t*>(extra + kPosOff)[pax * 256 + threadIdx.x % BT] = pw;
        wait_lds();
        turn_barrier();

        const int64_t extent = which == 0 ? p.mp : p.lp;
        T* __restrict__ out = static_cast<T*>(which == 0 ? p.qh : which == 1 ? p.k_out : p.vh);
        const int64_t tw = t0 + wt * Big<BT>::kWT;
        uint8_t* region = trans ? lds + wave * (Big<BT>::kWT * 256) : lds + Big<BT>::kSpare + wave * 2048;
        // + bias and the RMS, in place: feature tiles outside, so that each
        // parameter is read once
        float ss[NH][kTJ];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const f32x4 b4 = *reinterpret_cast<const f32x4*>(pb + i * 16 + h * 4);
#pragma unroll
            for (int j = 0; j < kTJ; ++j) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = bias != nullptr ? add_rn(acc[i][j][e], b4[e]) : acc[i][j][e];
                const float q = sum_sq<4>(v);
                ss[i / FPH][j] = i % FPH == 0 ? q : ss[i / FPH][j] + q;
                acc[i][j] = f32x4{v[0], v[1], v[2], v[3]};
            }
        }
        if (gamma != nullptr) {
#pragma unroll
            for (int hh = 0; hh < NH; ++hh)
#pragma unroll
                for (int j = 0; j < kTJ; ++j) {
                    float q = ss[hh][j];
                    q += __shfl_xor(q, 16);
                    q += __shfl_xor(q, 32);
                    ss[hh][j] = q < 1e-24f ? 1e12f : __builtin_amdgcn_rsqf(q);
                }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const f32x4 g4 = *reinterpret_cast<const f32x4*>(pg + i * 16 + h * 4);
#pragma unroll
                for (int j = 0; j < kTJ; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][e] = (acc[i][j][e] * ss[i / FPH][j]) * g4[e];
            }
        }
        // 16 tokens x 64 features at a time: RoPE, q's scale, pads, out
#pragma unroll
        for (int j = 0; j < kTJ; ++j) {
            const int64_t t = tw + j * 16 + fr;
            const int64_t tc = t < g.rows ? t : g.rows - 1;   // clamped for position reads
            const bool live = t < g.rows;
            f32x16 cs;
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                // cos/sin of the lane's slot pairs: cs[4 i ..] = (c, s) of slots s0 + i * 8, + 1
                // (both halves are whole heads of 64: the same slots)
                const int s0 = (FPH == 8 ? hf * 32 : 0) + h * 2;
                if (rope && (FPH == 8 || hf == 0)) {
                    const uint32_t* words = reinterpret_cast<const uint32_t*>(extra + kPosOff);
                    const uint32_t w0 = words[wt * Big<BT>::kWT + j * 16 + fr];
                    if (!lookup) {
                        const float* row = p.phases + (int64_t)w0 * HD + s0 * 2;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const f32x4 v = *reinterpret_cast<const f32x4*>(row + i * 16);
#pragma unroll
                            for (int e = 0; e < 4; ++e) cs[i * 4 + e] = v[e];
                        }
                    } else {
                        const uint32_t w1 = p.pos_dim > 1 ? words[256 + wt * Big<BT>::kWT + j * 16 + fr] : 0;
                        const int co[4] = {(int16_t)w0, (int16_t)w1, (int)w0 >> 16, (int)w1 >> 16};
                        bool in = true;
#pragma unroll
                        for (int ax = 0; ax < 4; ++ax) in = in && (uint32_t)co[ax] < (uint32_t)npos;
                        if (__all(in)) {
                            const uint32_t rowb = (uint32_t)fd * 8;
                            const uint32_t r0 = co[0] * rowb, r1 = co[1] * rowb, r2 = co[2] * rowb, r3 = co[3] * rowb;
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const u32x2 sw = *reinterpret_cast<const u32x2*>(extra + kSlotOff + (s0 + i * 8) * 4);
#pragma unroll
                                for (int q = 0; q < 2; ++q) {
                                    const uint32_t ax = sw[q] >> 16;
                                    const uint32_t ro = ax == 0 ? r0 : ax == 1 ? r1 : ax == 2 ? r2 : ax == 3 ? r3 : 0u;
                                    const float2 v =
                                        *reinterpret_cast<const float2*>(extra + tab_off + ro + (sw[q] & 0xFFFFu));
                                    cs[i * 4 + q * 2] = v.x;
                                    cs[i * 4 + q * 2 + 1] = v.y;
                                }
                            }
                        } else {
                            float pos[T2H_MAX_POS_DIM] = {(float)co[0], (float)co[1], (float)co[2], (float)co[3]};
                            if (co[0] == kFar || co[1] == kFar) {
                                PosSource{fresh(p.coords), p.coord_cols, fresh(p.grid_res), p.pos_dim}.get(tc, pos);
                                // waited for here: at its use, every token would wait for the stores in flight
#pragma unroll
                                for (int ax = 0; ax < T2H_MAX_POS_DIM; ++ax) asm volatile("" : "+v"(pos[ax]));
                            }
                            // rolled: unrolled, its sincosf calls crowd the registers of the path that is taken
#pragma unroll 1
                            for (int n = 0; n < 8; ++n) {
                                const int at = (s0 + (n >> 1) * 8 + (n & 1)) * 4;
                                const uint32_t ax = *reinterpret_cast<const uint32_t*>(extra + kSlotOff + at) >> 16;
                                const float fq = *reinterpret_cast<const float*>(extra + kFreqOff + at);
                                const float lo = ax & 1 ? pos[1] : pos[0], hi = ax & 1 ? pos[3] : pos[2];
                                float cv, sv;
                                sincosf(mul_rn(ax & 2 ? hi : lo, fq), &sv, &cv);
                                cs[2 * n] = ax & 4 ? 1.0f : cv;
                                cs[2 * n + 1] = ax & 4 ? 0.0f : sv;
                            }
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = acc[hf * 4 + i][j][e];
                    if (rope) {
                        rotate_pair(v[0], v[1], cs[i * 4], cs[i * 4 + 1]);
                        rotate_pair(v[2], v[3], cs[i * 4 + 2], cs[i * 4 + 3]);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float x = which == 0 ? mul_rn(v[e], p.q_scale) : v[e];
                        v[e] = live ? x : 0.0f;
                    }
                    u32x2 w;
                    w.x = Word<T>::pack(v);
                    w.y = Word<T>::pack(v + 2);
                    const int ch = i * 2 + (h >> 1);        // 16-byte chunk of the 64 features
                    const int row = j * 16 + fr;
                    uint8_t* dst = trans ? region + row * 256 + (((hf * 8 + ch) ^ stage_swz(row)) * 16)
                                         : region + fr * 128 + ((ch ^ swz(fr)) * 16);
                    *reinterpret_cast<u32x2*>(dst + (h & 1) * 8) = w;
                }
                if (!trans) {        // 64 features: a head of 64, or half of one of 128
                    wait_lds();
                    const int64_t zz = HD == 64 ? z + hf : z;
#pragma unroll
                    for (int it = 0; it < 2; ++it) {
                        const int r = it * 8 + (lane >> 3), ch = lane & 7;
                        const u32x4 w = *reinterpret_cast<const u32x4*>(region + r * 128 + ((ch ^ swz(r)) * 16));
                        const int64_t to = tw + j * 16 + r;
                        if (to < extent)
                            out_store16(out + (zz * extent + to) * HD + (HD == 64 ? 0 : hf * 64) + ch * 8, w);
                    }
                    wait_lds();
                }
            }
        }
        if (trans) {
            // feature rows of the transposed k: lane (d, gg) gathers feature d of
            // tokens 8 gg .. 8 gg + 7 (eight 2-byte reads, one per token row)
            constexpr int kG = Big<BT>::kWT / 8;
            wait_lds();
#pragma unroll 2
            for (int it = 0; it < kHead * kG / 64; ++it) {
                const int d = it * (64 / kG) + lane / kG;
                const int gg = lane % kG;
                const int off = (d & 7) * 2;
                u32x4 w;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int r0 = gg * 8 + 2 * q, r1 = r0 + 1;
                    const uint32_t lo = *reinterpret_cast<const uint16_t*>(
                        region + r0 * 256 + (((d >> 3) ^ stage_swz(r0)) * 16) + off);
                    const uint32_t hi = *reinterpret_cast<const uint16_t*>(
                        region + r1 * 256 + (((d >> 3) ^ stage_swz(r1)) * 16) + off);
                    w[q] = lo | (hi << 16);
                }
                const int64_t to = tw + gg * 8;
                if (to < extent) {
                    u32x4* dst = reinterpret_cast<u32x4*>(out + ((int64_t)z * HD + d) * p.lp + to);
                    if constexpr (BT == 256) __builtin_nontemporal_store(w, dst);    // whole lines
                    else *dst = w;
                }
            }
            wait_lds();
            turn_barrier();       // every wave has read its share of the stages
            if (next) c.prologue(steps);
        }
        if (!more) break;
    }
}

template <typename T, int HD, int BT, bool W64>
hipError_t qkv_typed(GemmArgs g, const PackArgs& p, const RopeSlots& tab, int64_t span, hipStream_t s) {
    g.nblocks = ((span + BT - 1) / BT) * g.ftiles;
    const dim3 grid = persistent_grid(g.nblocks), blk(kThreads);
    if (p.k_transposed) hipLaunchKernelGGL((qkv_pack_kernel<T, true, HD, BT, W64>), grid, blk, 0, s, g, p, tab);
    else hipLaunchKernelGGL((qkv_pack_kernel<T, false, HD, BT, W64>), grid, blk, 0, s, g, p, tab);
    return hipGetLastError();
}

// 128-token tiles when 256-token ones would occupy half of the CUs at most;
// 256 otherwise. us back to back, f16, 4608 features of K = 1536, with bias,
// RMS and RoPE from coordinates (without RMS and RoPE): 1,200 tokens 33.5 (26.4)
// on 180 tiles of 128, 45.8 (33.7) on 90 of 256; 2,369 tokens 47.6 (36.0) on
// 180 of 256, 60.4 (48.9) on 342 of 128. From 3,600 to 5,000 tokens 128 would be
// 3-8 % faster with RMS and RoPE, 2-3 % slower without.
template <typename T, int HD>
hipError_t qkv_sized(const GemmArgs& g, const PackArgs& p, const RopeSlots& tab, int64_t span, hipStream_t s) {
    if (g.ldx > kMaxStride32 || g.k > kMaxStride32) return qkv_typed<T, HD, 128, true>(g, p, tab, span, s);
    if ((span + 255) / 256 * g.ftiles * 2 <= device_cu_count()) return qkv_typed<T, HD, 128, false>(g, p, tab, span, s);
    return qkv_typed<T, HD, 256, false>(g, p, tab, span, s);
}

}  // namespace

bool gemm_head_dim_ok(int32_t head_dim) { return head_dim == 128 || head_dim == 64; }

hipError_t launch_qkv_pack(GemmArgs g, const PackArgs& p, const RopeSlots& tab, hipStream_t s) {
    // token tiles cover the pad rows of the outputs too (they are written as 0)
    int64_t span = g.rows;
    if (p.mp > span) span = p.mp;
    if (p.lp > span) span = p.lp;
    g.ftiles = g.n / kBF;
    g.tgroup = tile_group(g.k);
    if (span == 0) return hipSuccess;
    if (p.head_dim == 64) {
        if (g.dtype == T2H_F16) return qkv_sized<_Float16, 64>(g, p, tab, span, s);
        return qkv_sized<__bf16, 64>(g, p, tab, span, s);
    }
    if (g.dtype == T2H_F16) return qkv_sized<_Float16, 128>(g, p, tab, span, s);
    return qkv_sized<__bf16, 128>(g, p, tab, span, s);
}

}  // namespace t2h
