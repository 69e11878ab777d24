// Attention for wide heads, 128 < d <= 256 (d a multiple of 8), forward and backward on MFMA:
// fp32 on v_mfma_f32_32x32x2f32, bf16 / fp16 on v_mfma_f32_32x32x16_{bf16,f16}, gfx950.
//
// Same math as the generic kernels that take these head dims otherwise (attn_generic.hip;
// flash_attention.cu:97-161, :269-311), which hold P and dS in fp32.  The 16-bit MFMA takes
// 16-bit operands, so P and dS go in as a sum of terms, each the rounding to 16 bits of what
// the terms before it leave, one MFMA each into the same fp32 accumulator (the inputs are exact):
// three for bf16 (24 significant bits, as fp32), two for fp16 (22).  Share of outputs that are
// not the 64-bit result rounded once, B2 H8 T1024 d256 unmasked: bf16 generic 0.050-0.053 %, two
// terms 0.241-0.247 %, three 0.033-0.044 %; fp16 generic 0.42-0.46 %, two terms 0.18-0.25 %.
// The third bf16 term costs 10 % (forward and backward 214 -> 237 us).  fp16 has fp32's precision
// but not its range: P (<= 2^8) is scaled by a constant power of two, and dS by a running one per
// own row that follows the largest |dS| of the row, the accumulator rescaled when it grows (as the
// softmax rescales O).
//
// One kernel, four passes (MODE), all of one form: every lane owns one row of the "own"
// tensors, kept in registers as the B operand, and walks 32-row blocks of two "stream" tensors
// X and Y in LDS:
//            own1  own2   X  Y   out[own][:] += sum over stream rows
//   kFwd      Q     -     K  V   P  Y
//   kDq       Q     dO    K  V   dS X
//   kDk       K     V     Q  dO  dS X
//   kDv       K     -     Q  dO  P  Y
// S^T = X own1^T puts stream rows in accumulator registers and own rows in lanes, so P / dS
// are the B operands of out^T += Y^T P (X^T dS) without moving between lanes, and X^T / Y^T are
// read column-wise from the row-major tiles.  dK and dV are separate passes: one wave's
// registers hold 256 fp32 accumulators for one of them beside the own rows, not for both.
//
// A masked P or dS is 0, but 0 times an infinity or NaN of the tile is not, and the 16-bit split
// of an infinity is a NaN.  A wave whose result is not finite recomputes its 32 own rows one
// after another in scalar fp32, over the mask's positions only, as the generic kernels do.
//
// A workgroup has 4 waves.  16-bit: 64 own rows, 2 waves on even stream blocks and 2 on odd
// ones (each pair with its own double-buffered tiles, summed through LDS at the end): twice the
// workgroups of 128 rows, for grids of a few heads.  fp32: 128 own rows, tiles of twice the
// bytes shared by all four.  128 KB of tiles, one workgroup per CU, one wave per SIMD with up to
// 512 registers.  Bound: MFMA issue of one wave per SIMD, which its own exponentials and
// conversions interrupt; per 32 x 32 tile of the mask the passes execute, for the convention's
// 2 + 5 units, bf16 4 + 5 + 5 + 4, fp16 3 + 4 + 4 + 3 and fp32 2 + 3 + 3 + 2.  Measured, B2 H8
// T1024 d256 bf16 unmasked, forward and backward: generic kernels 60 700 us, this 237 (forward 49,
// preprocess 6, dQ 59, dK 66, dV 57; matrix cores busy 15 to 25 % of the launches).
#include "attn_bf16_tiles.h"
#include "attn_launch.h"

#include <math.h>

#include <type_traits>

namespace ctattn {
namespace {

using namespace bf16tile;

enum WideMode { kFwd, kDq, kDk, kDv };

// 16 zero bytes: the source of the tile columns d .. 32 NT - 1.
__device__ __attribute__((aligned(16))) const uint32_t wide_zeros[4] = {0, 0, 0, 0};

typedef __attribute__((address_space(3))) const float lds_cfloat;
typedef __attribute__((address_space(3))) float lds_float;
__device__ __forceinline__ float lds_f1(uint32_t addr) { return *(lds_cfloat *)(uintptr_t)addr; }
__device__ __forceinline__ void lds_st1(uint32_t addr, float x) { *(lds_float *)(uintptr_t)addr = x; }

// Storage formats.  A tile is 32 rows of 256 elements (whatever NT), the 16-byte chunk c of row
// r at physical chunk c ^ swz(r).  `row(tile, st)`: A operand of contraction step st over the
// head dim, from the lane's tile row; `cols`: the A operands of the contraction over the 32 tile
// rows for head-dim tile dt, in the row order of the accumulator registers.
template <typename F>
struct Wide16 {
    using Fmt = F;
    using Vec = typename F::vec;
    static constexpr bool WIDE = false;
    static constexpr bool RANGE = std::is_same_v<F, F16Fmt>;  // 16-bit exponent range to guard
    static constexpr int TERMS = RANGE ? 2 : 3;               // of P and dS (see the head of the file)
    static constexpr int EB = 2, CH = 32, GROUPS = 2, SLOTS = 2;
    static constexpr int STEPS_PER_TILE = 2;  // contraction steps per 32 head-dim columns
    static constexpr float kPscaleFwd = RANGE ? 64.f : 1.f, kPscaleBwd = RANGE ? 16384.f : 1.f;
    __device__ static constexpr int swz(int r) { return Tile<256>::swz(r); }
    struct Lane {
        uint32_t r, c0, c1;
        __device__ void init(int lane) {
            r = row_base<256>(0, lane & 31, lane >> 5);
            c0 = col_base<256>(0, 0, 0, lane);
            c1 = col_base<256>(0, 0, 1, lane);
        }
    };
    __device__ static Vec row(uint32_t tile, const Lane &l, int st) {
        return lds_b128<Vec>(tile + (l.r ^ uint32_t(st << 5)));
    }
    __device__ static Vec col(uint32_t tile, const Lane &l, int kk, int dt) {
        return read_col<256, Vec>(tile + l.c0, tile + l.c1, kk, dt);
    }
    __device__ static Vec own(const char *p) { return *reinterpret_cast<const Vec *>(p); }
    __device__ static floatx16 mma(Vec a, Vec b, floatx16 c) { return F::mfma(a, b, c); }
    __device__ static float load(const char *p) { return F::widen(*reinterpret_cast<const uint16_t *>(p)); }
    __device__ static void store(char *p, float x) { *reinterpret_cast<uint16_t *>(p) = F::bits(x); }
    __device__ static void store4(char *p, floatx4 x) {
        *reinterpret_cast<u16x4 *>(p) = u16x4{F::bits(x[0]), F::bits(x[1]), F::bits(x[2]), F::bits(x[3])};
    }
};
struct Wide32 {
    using Vec = floatx4;
    static constexpr bool WIDE = true, RANGE = false;
    static constexpr int EB = 4, CH = 64, GROUPS = 1, SLOTS = 4;
    static constexpr int STEPS_PER_TILE = 4;
    static constexpr float kPscaleFwd = 1.f, kPscaleBwd = 1.f;
    // A row read takes one chunk of 16 consecutive rows: swz makes them 16 distinct chunks mod 16
    // (64 banks).  A column read takes 32 consecutive columns (8 chunks, all moved alike).
    __device__ static constexpr int swz(int r) { return r & 15; }
    struct Lane {
        uint32_t r, c;
        __device__ void init(int lane) {
            const int col = lane & 31, h = lane >> 5;
            r = uint32_t(col * 1024 + ((h ^ swz(col)) << 4));
            c = uint32_t(4 * h * 1024 + (((col >> 2) ^ (4 * h)) << 4) + 4 * (col & 3));
        }
    };
    // Head-dim elements 8 st + 4 half + 0..3.
    __device__ static Vec row(uint32_t tile, const Lane &l, int st) { return lds_f4(tile + (l.r ^ uint32_t(st << 5))); }
    // Column 32 dt + col of tile row 8 g + 4 half + t.
    __device__ static float col(uint32_t tile, const Lane &l, int g, int t, int dt) {
        return lds_f1(tile + (l.c ^ uint32_t(((8 * dt) ^ (8 * (g & 1)) ^ t) << 4)) + uint32_t((8 * g + t) * 1024));
    }
    __device__ static Vec own(const char *p) { return *reinterpret_cast<const Vec *>(p); }
    __device__ static floatx16 mma(Vec a, Vec b, floatx16 c) {
#pragma unroll
        for (int t = 0; t < 4; ++t) c = mfma32x32x2(a[t], b[t], c);
        return c;
    }
    __device__ static float load(const char *p) { return *reinterpret_cast<const float *>(p); }
    __device__ static void store(char *p, float x) { *reinterpret_cast<float *>(p) = x; }
    __device__ static void store4(char *p, floatx4 x) { *reinterpret_cast<floatx4 *>(p) = x; }
};

template <typename E>
struct WideCfg {
    static constexpr int NW = E::GROUPS * E::SLOTS;
    static constexpr int OB = 32 * E::SLOTS;          // own rows per workgroup
    static constexpr int ROW = 256 * E::EB;
    static constexpr int TILE = 32 * ROW;
    static constexpr int TILES = E::GROUPS * 4 * TILE;  // X, Y, double-buffered, per group
    static constexpr int STATS = TILES;                 // per group and buffer: 32 LSE, 32 delta
    static constexpr int SLOW = STATS + E::GROUPS * 2 * 256;  // per wave: 64 floats of the scalar path
    static constexpr int LDS = SLOW + NW * kWave * 4;
    static constexpr int NL = 32 * E::CH / kWave / E::SLOTS;  // load instructions per wave and tile
    static_assert(NW == 4 && LDS <= 160 * 1024, "LDS of one workgroup");
};

struct WideArgs {
    const char *own1, *own2, *x, *y;
    const float *lse, *delta;  // backward passes
    char *out;
    float *lse_out;  // forward, may be null
    int T, BH, d, causal;
    float c;       // log2(e) / sqrt(d)
    float oscale;  // dQ, dK: 1 / sqrt(d); dV: 1
};

// Loads rows s0 .. s0 + 31 of a (batch, head)'s [T][d] tensor (row s0 at `block`, `rows` of them
// before the end) into a tile.  Rows past the end re-read the last one (masked later); PAD (d not
// a multiple of 32): chunks past d read zeros, so they add nothing to a contraction over d.  Whole
// 32-wide head-dim tiles past d are never read and load the row's last chunk.
template <typename E, bool PAD>
__device__ __forceinline__ void wide_load(uint32_t tile, const char *block, int rows, int row_bytes, int slot,
                                          int lane) {
    using C = WideCfg<E>;
#pragma unroll
    for (int i = 0; i < C::NL; ++i) {
        const int P = (slot * C::NL + i) * kWave + lane;
        const int r = P / E::CH;
        const int b = ((P % E::CH) ^ E::swz(r)) * 16;  // byte offset in the row
        const uint32_t off = uint32_t(min(r, rows - 1) * row_bytes + min(b, row_bytes - 16));
        const char *g = block + off;
        if (PAD && b >= row_bytes) g = reinterpret_cast<const char *>(wide_zeros);
        const uint32_t dst = __builtin_amdgcn_readfirstlane(tile + uint32_t((slot * C::NL + i) * kWave * 16));
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(dst)
                     : "memory", "m0");
    }
}

// acc[dt] += (tile^T)[32 dt ..][stream] p[stream] for the lane's 16 stream rows per half.
template <typename E, int NT>
__device__ __forceinline__ void wide_accumulate(floatx16 (&acc)[NT], uint32_t tile, const typename E::Lane &ln,
                                                const float (&p)[16]) {
    if constexpr (E::WIDE) {
        constexpr int NS = 16 * NT, AHEAD = 6;
        float a[8];
        auto rd = [&](int i) { return E::col(tile, ln, (i % 16) >> 2, i & 3, i / 16); };
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) a[i] = rd(i);
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            if (i + AHEAD < NS) a[(i + AHEAD) & 7] = rd(i + AHEAD);
            read_fence();
            acc[i / 16] = mfma32x32x2(a[i & 7], p[i % 16], acc[i / 16]);
        }
    } else {
        using V = typename E::Vec;
        using el = typename E::Fmt::elem;
        V w[E::TERMS][2];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float x = p[r];
#pragma unroll
            for (int t = 0; t < E::TERMS; ++t) {
                const el h = (el)x;
                w[t][r / 8][r % 8] = h;
                x -= (float)h;
            }
        }
        constexpr int NS = 2 * NT, AHEAD = 3;
        V a[4];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) a[i] = E::col(tile, ln, i / NT, i % NT);
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            if (i + AHEAD < NS) a[(i + AHEAD) & 3] = E::col(tile, ln, (i + AHEAD) / NT, (i + AHEAD) % NT);
            read_fence();
#pragma unroll
            for (int t = 0; t < E::TERMS; ++t) acc[i % NT] = E::mma(a[i & 3], w[t][i / NT], acc[i % NT]);
        }
    }
}

// One (own, stream) position of the mask: own and stream index in [0, T), causal key <= row.
template <int MODE>
__device__ __forceinline__ bool wide_valid(int own, int stream, int T, int causal) {
    constexpr bool own_rows = MODE == kFwd || MODE == kDq;
    return stream < T && (!causal || (own_rows ? stream <= own : own <= stream));
}

template <typename E, int NT, int MODE, bool PAD>
struct WidePass {
    using C = WideCfg<E>;
    using V = typename E::Vec;
    static constexpr int KS = E::STEPS_PER_TILE * NT;
    static constexpr bool TWO = MODE == kDq || MODE == kDk;  // needs dP = Y own2^T

    V o1[KS], o2[TWO ? KS : 1];
    floatx16 acc[NT];
    float m_run, l_run;    // kFwd: running max (log2 units) and this half's share of the denominator
    float lse2, ndelta;    // kDq: LSE log2(e) and -delta of the lane's row
    float es;              // RANGE, dS: the scale of the lane's row in the accumulator
    typename E::Lane ln;

    // One 32 x 32 tile of the wave; masked: it crosses the diagonal or the end of the sequence.
    __device__ __forceinline__ void block(uint32_t xt, uint32_t yt, uint32_t stats, int s0, int own, int half,
                                          bool masked, const WideArgs &p) {
        floatx16 s = zero16(), dp;
        if constexpr (MODE == kDk) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const floatx4 d4 = lds_f4(stats + 128 + 16 * half + 32 * g);
#pragma unroll
                for (int t = 0; t < 4; ++t) dp[4 * g + t] = -d4[t];
            }
        }
        if constexpr (MODE == kDq) {
#pragma unroll
            for (int r = 0; r < 16; ++r) dp[r] = ndelta;
        }
        constexpr int AHEAD = 3;
        V xa[4], ya[TWO ? 4 : 1];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            xa[i] = E::row(xt, ln, i);
            if constexpr (TWO) ya[i] = E::row(yt, ln, i);
        }
#pragma unroll
        for (int st = 0; st < KS; ++st) {
            if (st + AHEAD < KS) {
                xa[(st + AHEAD) & 3] = E::row(xt, ln, st + AHEAD);
                if constexpr (TWO) ya[(st + AHEAD) & 3] = E::row(yt, ln, st + AHEAD);
            }
            read_fence();
            s = E::mma(xa[st & 3], o1[st], s);
            if constexpr (TWO) dp = E::mma(ya[st & 3], o2[st], dp);
        }
        float w[16];  // P or dS of the lane's own row and stream rows acc_row(r, half)
        if constexpr (MODE == kFwd) {
            if (masked) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (!wide_valid<MODE>(own, s0 + acc_row(r, half), p.T, p.causal)) s[r] = -INFINITY;
            }
            // Against the running max first; the block max only when a lane's share of P exceeds
            // 2^8 (the max grew by up to 8 in log2 units, or the first block's infinities).
            float psum = 0.f;
            auto exps = [&]() __attribute__((always_inline)) {
                psum = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    w[r] = fast_exp2(fmaf(s[r], p.c, -m_run));
                    psum += w[r];
                }
            };
            exps();
            if (__any(!(psum <= 256.f))) {
                float mx = s[0];
#pragma unroll
                for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
                mx = max_xor32(mx) * p.c;
                if (__any(mx > m_run + 8.f)) {
                    const float m_new = fmaxf(m_run, mx);
                    const float resc = fast_exp2(m_run - m_new);
                    m_run = m_new;
                    l_run *= resc;
#pragma unroll
                    for (int dt = 0; dt < NT; ++dt) acc[dt] *= resc;
                }
                exps();
            }
            l_run += psum;
        } else {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                floatx4 l4;
                if constexpr (MODE != kDq) l4 = lds_f4(stats + 16 * half + 32 * g);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int r = 4 * g + t;
                    const float l2 = MODE == kDq ? lse2 : l4[t] * kLog2e;
                    float x = fast_exp2(fmaf(s[r], p.c, -l2));
                    if constexpr (TWO) x *= dp[r];
                    w[r] = x;
                }
            }
            if (masked) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (!wide_valid<MODE>(own, s0 + acc_row(r, half), p.T, p.causal)) w[r] = 0.f;
            }
        }
        if constexpr (E::RANGE) scale(w);
        wide_accumulate<E, NT>(acc, TWO ? xt : yt, ln, w);
    }

    // fp16 P / dS into the format's range (see the head of the file).  Each row by itself: a row past
    // T (kDk: scores of 0 against LSEs far below 0) may hold anything.
    __device__ __forceinline__ void scale(float (&w)[16]) {
        if constexpr (!TWO) {
#pragma unroll
            for (int r = 0; r < 16; ++r) w[r] *= MODE == kFwd ? E::kPscaleFwd : E::kPscaleBwd;
        } else {
            float mx = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, fabsf(w[r]));
            if (__any(mx * es > 16384.f)) {
                mx = max_xor32(mx);  // of the row's two lanes
                float f = 1.f;
                if (mx * es > 16384.f && mx < INFINITY) {
                    // es = 2^(8 - exponent of mx), from the exponent bits: |dS| es in [2^8, 2^9).
                    const int e = int(__float_as_uint(mx) >> 23) - 127;
                    const float es_new = __uint_as_float(uint32_t(min(8 - e, 100) + 127) << 23);
                    f = es_new / es;
                    es = es_new;
                }
#pragma unroll
                for (int dt = 0; dt < NT; ++dt) acc[dt] *= f;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) w[r] *= es;
        }
    }

    // One own row by the whole wave in scalar fp32: 64 stream rows at a time one per lane, then the
    // output columns lane, lane + 64, ... .  ws: 64 floats of LDS.
    __device__ __attribute__((noinline)) static void slow_row(int own, int64_t base, int64_t rbase, int row_bytes,
                                                             uint32_t ws, int lane, const WideArgs &p) {
        constexpr bool own_rows = MODE == kFwd || MODE == kDq;
        const char *o1r = p.own1 + base + int64_t(own) * row_bytes;
        const char *o2r = TWO ? p.own2 + base + int64_t(own) * row_bytes : nullptr;
        const int lo = p.causal && !own_rows ? own : 0, hi = p.causal && own_rows ? own + 1 : p.T;
        float out[4] = {0.f, 0.f, 0.f, 0.f}, m = -INFINITY, l = 0.f;
        for (int s0 = lo; s0 < hi; s0 += kWave) {
            const int s = s0 + lane;
            float x = MODE == kFwd ? -INFINITY : 0.f;
            if (s < hi) {
                const char *xr = p.x + base + int64_t(s) * row_bytes, *yr = p.y + base + int64_t(s) * row_bytes;
                float dot = 0.f, dp = 0.f;
                for (int b = 0; b < row_bytes; b += E::EB) {
                    dot += E::load(o1r + b) * E::load(xr + b);
                    if constexpr (TWO) dp += E::load(o2r + b) * E::load(yr + b);
                }
                x = dot * (p.c * kLn2);
                if constexpr (MODE != kFwd) {
                    const int row = own_rows ? own : s;
                    x = expf(x - p.lse[rbase + row]);
                    if constexpr (TWO) x *= dp - p.delta[rbase + row];
                }
            }
            float resc = 1.f;
            if constexpr (MODE == kFwd) {
                const float mn = fmaxf(m, wave_max(x));
                resc = m == -INFINITY ? 0.f : expf(m - mn);
                x = s < hi ? expf(x - mn) : 0.f;
                l = l * resc + wave_sum(x);
                m = mn;
            }
            lds_st1(ws + uint32_t(4 * lane), x);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const int n = min(hi - s0, kWave);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int c = lane + kWave * k;
                if (c >= p.d) continue;
                out[k] *= resc;
                const char *z = (TWO ? p.x : p.y) + base + int64_t(s0) * row_bytes + c * E::EB;
                for (int j = 0; j < n; ++j) out[k] += lds_f1(ws + uint32_t(4 * j)) * E::load(z + int64_t(j) * row_bytes);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int c = lane + kWave * k;
            if (c < p.d)
                E::store(p.out + base + int64_t(own) * row_bytes + c * E::EB, MODE == kFwd ? out[k] / l : out[k] * p.oscale);
        }
        if constexpr (MODE == kFwd)
            if (p.lse_out != nullptr && lane == 0) p.lse_out[rbase + own] = m + logf(l);
    }

    __device__ void run(char *smem, const WideArgs &p) {
        const uint32_t L = lds_addr(smem);
        const int lane = threadIdx.x & (kWave - 1);
        const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
        const int group = wave / E::SLOTS, slot = wave % E::SLOTS;
        const int half = lane >> 5;
        constexpr bool own_rows = MODE == kFwd || MODE == kDq;
        const int T = p.T;
        const int id = blockIdx.x, bh = id % p.BH, nb = (T + C::OB - 1) / C::OB;
        // Longest first when causal: the last query block, the first key block.
        const int ob = p.causal && own_rows ? nb - 1 - id / p.BH : id / p.BH;
        const int w0 = ob * C::OB + 32 * slot, own = w0 + (lane & 31);
        const int row_bytes = p.d * E::EB;
        const int64_t base = int64_t(bh) * T * row_bytes, rbase = int64_t(bh) * T;
        ln.init(lane);

        const int first = p.causal && !own_rows ? ob * C::OB / 32 : 0;
        const int end = ((p.causal && own_rows ? min(T, (ob + 1) * C::OB) : T) + 31) / 32;
        const int iters = (end - first + E::GROUPS - 1) / E::GROUPS;
        const uint32_t mine = L + uint32_t(group * 4 * C::TILE);
        const uint32_t stats = L + uint32_t(C::STATS + group * 512);
        auto issue = [&](int sb, int buf) {
            const int s0 = 32 * sb;
            const int64_t off = base + int64_t(s0) * row_bytes;
            wide_load<E, PAD>(mine + uint32_t(buf * 2 * C::TILE), p.x + off, T - s0, row_bytes, slot, lane);
            wide_load<E, PAD>(mine + uint32_t((buf * 2 + 1) * C::TILE), p.y + off, T - s0, row_bytes, slot, lane);
            if constexpr (!own_rows) {
                if (slot == 0)
                    load_dword_dma((half ? p.delta : p.lse) + rbase + min(s0 + (lane & 31), T - 1),
                                   stats + uint32_t(buf * 256));
            }
        };
        if (first + group < end) issue(first + group, 0);

        // Own rows past T are zeros; nothing of them is stored.
        const int kb = 16 * half;  // bytes of the step this half supplies
#pragma unroll
        for (int st = 0; st < KS; ++st) {
            const int b = 32 * st + kb;
            o1[st] = V{};
            if (own < T && b < row_bytes) o1[st] = E::own(p.own1 + base + int64_t(own) * row_bytes + b);
            if constexpr (TWO) {
                o2[st] = V{};
                if (own < T && b < row_bytes) o2[st] = E::own(p.own2 + base + int64_t(own) * row_bytes + b);
            }
        }
        if constexpr (MODE == kDq) {
            lse2 = own < T ? p.lse[rbase + own] * kLog2e : 0.f;
            ndelta = own < T ? -p.delta[rbase + own] : 0.f;
        }
        m_run = -INFINITY;
        l_run = 0.f;
        es = 0x1p100f;
#pragma unroll
        for (int dt = 0; dt < NT; ++dt) acc[dt] = zero16();
        // The compiler's own loads above share vmcnt with the tile loads; wait for both once.
        for (int it = 0; it < iters; ++it) {
            const int sb = first + it * E::GROUPS + group, buf = it & 1;
            // This wave's loads of `buf` have landed; after the barrier every wave's have, and no
            // wave reads buf ^ 1 any more.
            wait_loads();
            lds_barrier();
            if (sb + E::GROUPS < end) issue(sb + E::GROUPS, buf ^ 1);
            const int s0 = 32 * sb;
            if (sb >= end || w0 >= T || (p.causal && (own_rows ? s0 > w0 + 31 : s0 + 31 < w0))) continue;
            const uint32_t xt = mine + uint32_t(buf * 2 * C::TILE), yt = xt + uint32_t(C::TILE);
            const uint32_t st = stats + uint32_t(buf * 256);
            const bool masked = s0 + 32 > T || (p.causal && (own_rows ? s0 + 31 > w0 : s0 < w0 + 31));
            block(xt, yt, st, s0, own, half, masked, p);
        }

        float os = p.oscale;
        if constexpr (MODE == kDv) os /= E::kPscaleBwd;
        if constexpr (TWO && E::RANGE) os /= es;
        if constexpr (MODE == kFwd) l_run += __shfl_xor(l_run, 32, kWave);
        if constexpr (E::GROUPS == 2) {
            // Group 1's state through LDS (the tiles are no longer read) into group 0's.
            constexpr int NR = NT * 16 + 2;
            static_assert(E::SLOTS * NR * kWave * 4 <= C::LDS, "merge buffer");
            float *mb = reinterpret_cast<float *>(smem) + slot * NR * kWave + lane;
            if constexpr (MODE != kFwd) {
#pragma unroll
                for (int dt = 0; dt < NT; ++dt) acc[dt] *= os;
            }
            __syncthreads();
            if (group == 1) {
#pragma unroll
                for (int dt = 0; dt < NT; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) mb[(dt * 16 + r) * kWave] = acc[dt][r];
                mb[(NR - 2) * kWave] = m_run;
                mb[(NR - 1) * kWave] = l_run;
            }
            __syncthreads();
            if (group == 1) return;
            float a0 = 1.f, a1 = 1.f;
            if constexpr (MODE == kFwd) {
                // An empty group 1 has m = -inf: weight 0 (group 0 always holds key 0).
                const float m1 = mb[(NR - 2) * kWave], l1 = mb[(NR - 1) * kWave];
                const float m = fmaxf(m_run, m1);
                a0 = fast_exp2(m_run - m);
                a1 = fast_exp2(m1 - m);
                m_run = m;
                l_run = l_run * a0 + l1 * a1;
            }
#pragma unroll
            for (int dt = 0; dt < NT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[dt][r] = acc[dt][r] * a0 + mb[(dt * 16 + r) * kWave] * a1;
            os = 1.f;
        }
        if constexpr (MODE == kFwd) os = 1.f / (l_run * E::kPscaleFwd);
        float z = MODE == kFwd ? 0.f * m_run + 0.f * l_run : 0.f;
#pragma unroll
        for (int dt = 0; dt < NT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) z = fmaf(acc[dt][r], 0.f, z);
        if (__any(own < T && !(z == 0.f))) {
            const uint32_t ws = L + uint32_t(C::SLOW + wave * kWave * 4);
#pragma unroll 1
            for (int i = w0; i < min(w0 + 32, T); ++i) slow_row(i, base, rbase, row_bytes, ws, lane, p);
            return;
        }
        if (own >= T) return;
        char *dst = p.out + base + int64_t(own) * row_bytes;
#pragma unroll
        for (int dt = 0; dt < NT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int c = 32 * dt + 8 * g + 4 * half;
                if (c >= p.d) continue;
                floatx4 x;
#pragma unroll
                for (int t = 0; t < 4; ++t) x[t] = acc[dt][4 * g + t] * os;
                E::store4(dst + c * E::EB, x);
            }
        if constexpr (MODE == kFwd)
            if (p.lse_out != nullptr && half == 0) p.lse_out[rbase + own] = (m_run + log2f(l_run)) * kLn2;
    }
};

template <typename E, int NT, int MODE, bool PAD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void wide_attn_kernel(WideArgs p) {
    __shared__ __attribute__((aligned(1024))) char smem[WideCfg<E>::LDS];
    WidePass<E, NT, MODE, PAD> pass;
    pass.run(smem, p);
}

template <typename E, int MODE>
hipError_t launch_wide(const WideArgs &p, int64_t bh, hipStream_t stream) {
    using C = WideCfg<E>;
    const int64_t blocks = (int64_t(p.T) + C::OB - 1) / C::OB * bh;
    if (!grid_fits(blocks, 256)) return hipErrorInvalidValue;
    const dim3 grid{unsigned(blocks)}, block{256};
    // 32-column head-dim tiles: 5 or 6 of them for d = 160 and 192, else all 8 (136 and 224 too: every
    // count is another four kernels a type to build).
    if (p.d == 160)
        hipLaunchKernelGGL((wide_attn_kernel<E, 5, MODE, false>), grid, block, 0, stream, p);
    else if (p.d == 192)
        hipLaunchKernelGGL((wide_attn_kernel<E, 6, MODE, false>), grid, block, 0, stream, p);
    else if (p.d == 256)
        hipLaunchKernelGGL((wide_attn_kernel<E, 8, MODE, false>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((wide_attn_kernel<E, 8, MODE, true>), grid, block, 0, stream, p);
    return hipGetLastError();
}

template <typename E>
hipError_t wide_fwd(const void *q, const void *k, const void *v, void *o, float *lse, const AttnShape &s,
                    hipStream_t stream) {
    WideArgs p{};
    p.own1 = static_cast<const char *>(q);
    p.x = static_cast<const char *>(k);
    p.y = static_cast<const char *>(v);
    p.out = static_cast<char *>(o);
    p.lse_out = lse;
    p.T = int(s.T);
    p.BH = int(s.bh());
    p.d = int(s.d);
    p.causal = s.causal;
    p.c = kLog2e / sqrtf(float(s.d));
    p.oscale = 1.f;
    return launch_wide<E, kFwd>(p, s.bh(), stream);
}

template <typename E>
hipError_t wide_bwd(const void *q, const void *k, const void *v, const void *dout, const float *lse,
                    const float *delta, void *dq, void *dk, void *dv, const AttnShape &s, hipStream_t stream) {
    WideArgs p{};
    p.T = int(s.T);
    p.BH = int(s.bh());
    p.d = int(s.d);
    p.causal = s.causal;
    p.c = kLog2e / sqrtf(float(s.d));
    p.oscale = 1.f / sqrtf(float(s.d));
    p.lse = lse;
    p.delta = delta;
    // Own: query rows.
    p.own1 = static_cast<const char *>(q);
    p.own2 = static_cast<const char *>(dout);
    p.x = static_cast<const char *>(k);
    p.y = static_cast<const char *>(v);
    p.out = static_cast<char *>(dq);
    hipError_t e = launch_wide<E, kDq>(p, s.bh(), stream);
    if (e != hipSuccess) return e;
    // Own: keys.
    p.own1 = static_cast<const char *>(k);
    p.own2 = static_cast<const char *>(v);
    p.x = static_cast<const char *>(q);
    p.y = static_cast<const char *>(dout);
    p.out = static_cast<char *>(dk);
    e = launch_wide<E, kDk>(p, s.bh(), stream);
    if (e != hipSuccess) return e;
    p.oscale = 1.f;
    p.out = static_cast<char *>(dv);
    return launch_wide<E, kDv>(p, s.bh(), stream);
}

}  // namespace

// Shortest sequences worth a 32 x 32 tile: below them one wave per row (the generic kernels) is
// faster.  Measured, us, wide / generic, B H T at d = 256 causal: bf16 backward 1 1 1 47.5 / 42.3,
// 4 8 16 52.6 / 63.1, 32 32 8 188 / 281; fp32 forward 1 1 16 20.3 / 26.5, 32 32 8 85 / 69,
// backward 1 2 64 142 / 123, 1 4 128 249 / 273 (on eight tiles the fp32 dQ, dK and forward spill 201,
// 221 and 40 registers: two sets of own rows are 256 of them; fp16 dK spills 26, the other passes none).
bool wide_supported(int dtype, const AttnShape &s, bool backward) {
    const int64_t min_t = dtype != 0 ? 8 : backward ? 96 : 32;
    return (dtype == 0 || dtype == 1 || dtype == 2) && s.d > 128 && s.d <= 256 && s.d % 8 == 0 && s.T >= min_t &&
           s.T <= (int64_t(1) << 30) && grid_fits((s.T + 63) / 64 * s.bh(), 256);
}

hipError_t launch_wide_fwd(int dtype, const void *q, const void *k, const void *v, void *o, float *lse,
                           const AttnShape &s, hipStream_t stream) {
    return dtype == 0   ? wide_fwd<Wide32>(q, k, v, o, lse, s, stream)
           : dtype == 1 ? wide_fwd<Wide16<Bf16Fmt>>(q, k, v, o, lse, s, stream)
                        : wide_fwd<Wide16<F16Fmt>>(q, k, v, o, lse, s, stream);
}

hipError_t launch_wide_bwd(int dtype, const void *q, const void *k, const void *v, const void *o, const void *dout,
                           const float *lse, float *delta, void *dq, void *dk, void *dv, const AttnShape &s,
                           hipStream_t stream) {
    const hipError_t e = launch_bwd_preprocess(dtype, o, dout, delta, s, stream);
    if (e != hipSuccess) return e;
    return dtype == 0   ? wide_bwd<Wide32>(q, k, v, dout, lse, delta, dq, dk, dv, s, stream)
           : dtype == 1 ? wide_bwd<Wide16<Bf16Fmt>>(q, k, v, dout, lse, delta, dq, dk, dv, s, stream)
                        : wide_bwd<Wide16<F16Fmt>>(q, k, v, dout, lse, delta, dq, dk, dv, s, stream);
}

}  // namespace ctattn
