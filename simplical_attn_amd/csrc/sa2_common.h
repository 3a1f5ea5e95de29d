// Shared declarations of the gfx950 2-simplicial attention kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sa2.h"

namespace sa2 {

// One [B,N,H,D] tensor: base pointer and element strides (D stride is 1).
struct Tensor {
    void* p;
    int64_t sb, sn, sh;
    __host__ __device__ int64_t off(int b, int n, int h) const { return b * sb + n * sn + h * sh; }
};

// Everything a kernel needs about one call.  w1/w2 are already the inclusive
// window reaches: query i sees keys [i-w, i].
struct Problem {
    int B, N, H, D;
    int w1, w2;
    float scale, k2_bias, v2_bias;
    Tensor q, k1, k2, v1, v2, out, dout;
    Tensor dq, dk1, dk2, dv1, dv2;   // p == nullptr: not requested
    float* lse;                      // [B,H,N]
    float* dsum;                     // [B,H,N]  sum_d dout*out
    void* scratch;                   // remaining workspace (path specific)
    size_t scratch_bytes;
    size_t room;                     // backward: bytes the plans may spend on partial sums (ROOM_ANY: what they think best)
    int nsplit;                      // forward: shares of the rounds (partial outputs in `scratch` when more than one)
    int force_prepass;               // take the pre-pass kernels whenever the window allows, whatever the size
};

// ---- element loads / stores -------------------------------------------------
struct bf16_t { uint16_t bits; };
struct f16_t { _Float16 v; };

__device__ __forceinline__ float to_float(float x) { return x; }
__device__ __forceinline__ float to_float(bf16_t x) { return __uint_as_float(((uint32_t)x.bits) << 16); }
__device__ __forceinline__ float to_float(f16_t x) { return (float)x.v; }

__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);   // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);                                             // round to nearest even
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ void from_float(float f, float* p) { *p = f; }
__device__ __forceinline__ void from_float(float f, bf16_t* p) { p->bits = f32_to_bf16_bits(f); }
__device__ __forceinline__ void from_float(float f, f16_t* p) { p->v = (_Float16)f; }

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Workgroups are dealt round-robin to the 8 XCDs, each with its own L2: gives every XCD a run of consecutive work items,
// so that neighbours in the problem (which share most of their K/V window) meet in one L2.  A permutation of
// 0 .. total-1 for every total.
__device__ __forceinline__ int xcd_order(int pid, int total) {
    const int x = pid & 7, each = total >> 3, more = total & 7;
    return x * each + (x < more ? x : more) + (pid >> 3);
}

// log(sum_w + 1e-8) from the running maximum m and l = sum exp(s-m), for any m.
__device__ __forceinline__ float lse_with_eps(float m, float l) {
    const float log_eps = -18.420680743952367f;   // log(1e-8)
    if (m > log_eps) return m + logf(l + 1e-8f * expf(-m));
    return log_eps + log1pf(l * expf(m - log_eps));
}

// Lifts a kernel's limit on dynamic LDS to the CU's full 160 KB.  The value never depends on the
// call, and it is set once per (kernel, device) for the life of the process, so concurrent
// launches of one kernel with different LDS sizes cannot disturb each other.
constexpr int LDS_BYTES_PER_CU = 160 * 1024;
bool allow_full_lds(const void* kernel);

// ---- how a launch divides its work ------------------------------------------
// The kernels keep one workgroup per CU, so a grid runs in waves of 256 workgroups: every whole wave takes the mean
// workgroup's time, what is left over mostly the longest's, and the grid ends no sooner than that one.  Where a grid is
// smaller than the chip, or its last wave nearly empty, or its workgroups uneven (short ones at the ends of the
// sequence), the plans below cut the work of a workgroup into shares with fp32 partial sums, which cost their write and
// read (2.5 MB per unit of time, a sweep step of about 1 us) and a summation launch.  The constants are the ones whose
// choices lost least against the best of up to sixteen measured cuts (2.6 % on average for the K'-side kernel at nineteen
// sizes; the 16-bit K-side kernel has its own, see kv_plan).  In 16 bits they were measured with paired wavefronts on the K' side and
// one unit per wavefront in the forward, and hold for what runs there now as far as its times are alike.  All plans depend on
// the problem's sizes only.
constexpr int CUS = 256;
inline double grid_time(int64_t workgroups, double longest, double mean) {
    const int64_t waves = workgroups / CUS;
    const double t = (double)waves * mean + (workgroups - waves * CUS > 2 ? 0.7 * longest + 0.3 * mean : 0.0);
    return t > longest ? t : longest;
}
// mean over the sequence of min(i, w) / w
inline double window_fill(int w, int N) { return w < N ? 1.0 - 0.5 * w / N : 0.5 * N / w; }
constexpr double PART_BYTES_PER_STEP = 2.5e6, SUM_LAUNCH_STEPS = 8;

// All partial sums of a call that has to make do with `room` bytes: the plans cut less, down to the uncut launch
constexpr size_t ROOM_ANY = ~(size_t)0;
inline size_t room_left(size_t room, size_t taken) { return room == ROOM_ANY ? room : room > taken ? room - taken : 0; }

// The K' window in nseg segments of segw deltas, one workgroup per (K' block, segment)
struct KpPlan {
    int segw, nseg;
};
// The uncut launch's pre-pass (the single delta over of w2 = 4n) is charged as the round it saves: at B1 H16 N8192 D128
// w 512/32 eight rounds and the pre-pass take 2826 us, nine rounds (w 512/33) 2895.
// Segments are whole rounds of `upr` deltas, at most `most` deltas (what LDS holds).  A round sweeps the tiles of the K
// window; the work between two sweeps takes about two tiles' time, or five and a half where the rows of q and dO do not
// fit LDS beside the accumulator (raw(segment)), prologue and epilogue about eight.  bytes(plan): all partial sums; a cut may
// take 32 MiB, or three times what the uncut launch needs.
// Measured on the 16-bit kernel (us, uncut -> planned): B2 H4 N512 D64 w 256/256 607 -> 234 (seven segments),
// B3 H21 N282 D128 w 176/48 488 -> 303 (three), B1 H8 N4096 D128 w 128/64 862 -> 655 (two: the rows then fit LDS),
// B2 H4 N256 D64 w 32/32 43 -> 29 (three), B1 H8 N32768 D128 w 1024/64 19809 -> 19385 (two; 0.66 GB more of partial sums).
// Against every cut (profiles/plan_cuts.md): the plane-split kernels within 3.0 % of the best at ten sizes, head_dim 256
// within 3.2 % at seven of eight (27 % off at B1 H3 N700 w 500/100, where the bytes bind), the 16-bit kernels within 0.2 % at
// ten of twelve (30 % off at B4 H8 N2048 D128 w 64/48, 6 % at B4 H16 N2048 D128 w 1024/96).
template <class Raw, class Bytes>
KpPlan plan_segments(int B, int N, int H, int w1, int w2, int upr, int most, size_t room, Raw&& raw, Bytes&& bytes) {
    constexpr int ROWS = 32, MOST_SEGMENTS = 16;
    const int64_t base = (int64_t)B * H * ((N + ROWS - 1) / ROWS);
    const int rounds = (w2 + upr) / upr;
    const double tiles = ((w1 < N ? w1 : N) + ROWS + upr) / (double)ROWS + 1, fill = window_fill(w1, N) * window_fill(w2, N);
    KpPlan best = most > w2 ? KpPlan{w2 + 1, 1} : KpPlan{most, (w2 + most) / most};
    const double first_bytes = (double)bytes(best), likes = 3 * first_bytes > 33554432.0 ? 3 * first_bytes : 33554432.0;
    const double cap = likes < (double)room ? likes : (double)room;
    double least = 0;
    for (int nseg = best.nseg, last = 0; nseg <= MOST_SEGMENTS || least == 0; ++nseg) {
        const int per = (rounds + nseg - 1) / nseg;                                  // rounds per segment
        if (per == last || per < 1) continue;
        last = per;
        const KpPlan pl = least == 0 ? best : KpPlan{per * upr, (rounds + per - 1) / per};
        const double part = (double)bytes(pl);
        if (least != 0 && part > cap) break;
        const double sweep = per * (tiles + (raw(pl.segw) ? 2.0 : 5.5));
        const double cost = grid_time(base * pl.nseg, sweep + 8, sweep * fill + 8) + part / PART_BYTES_PER_STEP;
        if (least == 0 || cost < least) {
            least = cost;
            best = pl;
        }
        if (per == 1) break;
    }
    return best;
}

inline size_t fwd_part_bytes(int B, int N, int H, int width, int nsplit) {
    return nsplit > 1 ? (size_t)nsplit * B * H * (size_t)N * (width + 2) * sizeof(float) : 0;
}
// A forward launch in nsplit shares of the rounds of `upr` deltas: fp32 partial outputs in the workspace.  A round takes
// about three tiles' time beside its sweep, prologue and epilogue about eight.  Against every cut: the best or within 2 % at eight of
// fifteen sizes, 5 - 25 % off at the others, where a grid a little under a whole wave would take more shares.
// Two or three rounds are shared only where all shares run at once, a workgroup per CU, and save more than the merging launch costs
// (`least_saved` tiles of a sweep, by how long a kernel takes for one): fp32 B1 H2 N128 D64 w 32/16 26.3 -> 18.2 us, bf16
// B1 H4 N512 w 64/20 D96 31.4 -> 20.9, D128 25.2 -> 18.8, D256 36.9 -> 30.9, D64 w 200/12 20.7 -> 17.5, but w 40/8 12.2 -> 14.4, w 63/17 13.6 -> 13.8; not all at once: B1 H8
// N1024 D96 w 128/16 36.3 -> 57.4.  They stay one launch where the caller's workspace, `room`, has no place for them.
inline int plan_forward(int B, int N, int H, int width, int w1, int w2, int upr, int least_saved, size_t room) {
    constexpr int ROWS = 32, MOST = 16;
    const int64_t rows = (int64_t)B * H * N, base = (int64_t)B * H * ((N + ROWS - 1) / ROWS);
    const int rounds = ((w2 < N - 1 ? w2 : N - 1) + upr) / upr;
    const double tiles = ((w1 < N ? w1 : N) + ROWS) / (double)ROWS + 1;
    if (rounds < 4) {
        for (int ns = rounds; ns > 1; --ns)
            if (base * ns <= CUS && (rounds - (rounds + ns - 1) / ns) * tiles >= least_saved)
                return fwd_part_bytes(B, N, H, width, ns) <= room ? ns : 1;
        return 1;
    }
    if (base >= 3 * CUS) return 1;
    const double fill = window_fill(w1, N) * window_fill(w2, N);
    int best = 1;
    double least = 0;
    for (int ns = 1, last = 0; ns <= MOST && ns <= rounds; ++ns) {
        const int per = (rounds + ns - 1) / ns;
        if (per == last) continue;
        last = per;
        const int shares = (rounds + per - 1) / per;
        const double part = shares > 1 ? (double)shares * rows * (width + 2) * 4 : 0;
        if (part > 67108864.0) break;
        const double sweep = per * (tiles + 3);
        const double cost = grid_time(base * shares, sweep + 8, sweep * fill + 8) + (shares > 1 ? SUM_LAUNCH_STEPS + part / PART_BYTES_PER_STEP : 0);
        if (least == 0 || cost < 0.95 * least) {
            least = cost;
            best = shares;
        }
    }
    return best;
}

// ---- launchers (each returns a sa2_status) ----------------------------------
int launch_rowdot(const Tensor& out, const Tensor& dout, float* dsum, int B, int N, int H, int D,
                  int dtype, hipStream_t st);
int launch_generic_fwd(const Problem& p, int dtype, hipStream_t st);
int launch_generic_bwd(const Problem& p, int dtype, hipStream_t st);
size_t generic_bwd_scratch_bytes(int B, int N, int H, int D, int w1, int w2);

bool mfma_supported(int B, int N, int H, int D, int w1, int w2, int dtype);
bool mfma_bwd_supported(int B, int N, int H, int D, int w1, int w2, int dtype);
bool mfma_layout_ok(const Problem& p, bool backward);
int launch_mfma_fwd(const Problem& p, int dtype, hipStream_t st);
int mfma_fwd_nsplit(int B, int N, int H, int D, int w1, int w2, bool force_prepass, size_t room);
size_t mfma_fwd_part_bytes(int B, int N, int H, int D, int nsplit);
int launch_mfma_bwd(const Problem& p, int dtype, hipStream_t st);
size_t mfma_bwd_scratch_bytes(int B, int N, int H, int D, int w1, int w2, size_t room);
// fp32 arithmetic on the 16-bit MFMA, operands as sums of bf16 planes (sa2_split_mfma.hip): fp32 tensors of any head_dim up to 128 that is a multiple of 4, and 16-bit tensors
// of the head dims the 16-bit kernels do not have (multiples of 8 up to 120); rows 16-byte aligned
bool f32_mfma_supported(int D, int dtype);
bool f32_mfma_bwd_supported(int D, int w2, int dtype);
bool f32_mfma_layout_ok(const Problem& p, int dtype, bool backward);
size_t f32_mfma_bwd_scratch_bytes(int B, int N, int H, int D, int w1, int w2, int dtype, size_t room);
int launch_f32_mfma_fwd(const Problem& p, int dtype, hipStream_t st);
int f32_mfma_fwd_nsplit(int B, int N, int H, int D, int w1, int w2, int dtype, size_t room);
size_t f32_mfma_fwd_part_bytes(int B, int N, int H, int D, int nsplit);
int split_fwd_route(int B, int N, int H, int D, int w1, int w2, int dtype);
int split_kp_route(int B, int N, int H, int D, int w1, int w2, int dtype);
int split_kv_route(int B, int N, int H, int D, int w1, int w2, int dtype);
int launch_f32_mfma_bwd(const Problem& p, int dtype, hipStream_t st);
// Its forward and K side with one wavefront per SIMD (sa2_split_fwd_lone.h, sa2_split_kv_lone.h).  `width`: of the kernel; `two_planes`:
// products of a unit have 16 bits
int launch_split_fwd_lone_bf16(const Problem& p, int width, bool two_planes, hipStream_t st);
int launch_split_fwd_lone_fp16(const Problem& p, int width, bool two_planes, hipStream_t st);
int launch_split_fwd_lone_fp32(const Problem& p, int width, bool two_planes, hipStream_t st);
int launch_split_kv_lone_bf16(const Problem& p, int width, bool two_planes, int nsplit, float* part, hipStream_t st);
int launch_split_kv_lone_fp16(const Problem& p, int width, bool two_planes, int nsplit, float* part, hipStream_t st);
int launch_split_kv_lone_fp32(const Problem& p, int width, bool two_planes, int nsplit, float* part, hipStream_t st);
// 16-bit tensors with head_dim 256 on the 16-bit MFMA (rows 16-byte aligned)
bool wide_supported(int D, int dtype);
bool wide_bwd_supported(int D, int w2, int dtype);
size_t wide_bwd_scratch_bytes(int B, int N, int H, int D, int w1, int w2, size_t room);
int wide_fwd_nsplit(int B, int N, int H, int w1, int w2, size_t room);
int launch_wide_fwd(const Problem& p, int dtype, hipStream_t st);
int launch_wide_bwd(const Problem& p, int dtype, hipStream_t st);
// Partial outputs of a split forward, [nsplit][B*H*N] pairs (reference exponent M, sum L) and then
// [nsplit][B*H*N][width] sums at that reference, merged into out and lse in share order
int launch_fwd_merge(const Problem& p, int width, int dtype, hipStream_t st);
// K'-side backward kernel (dQ, dK', dV') that keeps its partial sums on chip (K' windows too wide for
// that are cut into segments of deltas, one workgroup each)
size_t kp_scratch_bytes(int B, int N, int H, int D, int w1, int w2, size_t room);
// Where the two kernels leave fp32 partial sums, rows of the kernel's width: the dQ partials of (K' block, segment)
// workgroups, [dV' | dK'][kp_n][B*H][N][width] of a segmented K'-side launch and [dK | dV][kv_n][B*H][N][width] of a split
// K-side launch.  NULL: that kernel wrote its results itself (dQ: not wanted).
struct BwdSums {
    const float *dq, *kp, *kv;
    int nkb, nseg, segw, kp_n, kv_n;
};
int launch_bwd_sums(const Problem& p, const BwdSums& sums, int width, int dtype, hipStream_t st);
int launch_mfma_bwd_kp(const Problem& p, int dtype, hipStream_t st, BwdSums* sums);
// What a 16-bit launch is made of, for tests that are about one kernel: bit 0 the pre-pass runs, bit 1 the main kernel is the
// one of sa2_mfma_fwd_lone.h or sa2_mfma_bwd_kp_lone.h, from bit 8 on shares or segments (K side: bits 0-7 K blocks per wavefront)
int mfma_fwd_route(int B, int N, int H, int head_dim, int w1, int w2, bool force_prepass);
int mfma_kp_route(int B, int N, int H, int head_dim, int w1, int w2, bool force_prepass);
int mfma_kv_route(int B, int N, int H, int head_dim, int w1, int w2);
// K-side backward kernel (dK, dV), one wavefront per SIMD; for small grids it splits a key block's stream of
// units over several workgroups, whose fp32 partial sums lie in the workspace behind the
// K'-side part (kp_side_scratch_bytes); K' windows too wide for its LDS rows are walked in segments
size_t kv_split_scratch_bytes(int B, int N, int H, int D, int w1, int w2, size_t room);
size_t kp_side_scratch_bytes(int B, int N, int H, int D, int w1, int w2, size_t room);
int launch_mfma_bwd_kv(const Problem& p, int dtype, hipStream_t st, BwdSums* sums);

}  // namespace sa2
