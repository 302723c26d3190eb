// gdn_chunked.hip -- chunked Gated DeltaNet prefill for gfx950 (fp16 MFMA, fp32 state).
//
// Chunk algebra (the chunk structure of gdn_chunked_cpu, src/gdn_sm75.cu:1109-1244, with
// the exact inverse).  Per V-head and chunk of C = 64 tokens, rows = tokens t, with
// G_t = in-chunk inclusive cumsum of g_log:
//   A[t][s]   = beta_t (k_t . k_s) e^{G_t - G_s}      s < t        (strictly lower)
//   T'        = (I + A)^-1 diag(beta)
//   Aqk[t][s] = (q_t . k_s) e^{G_t - G_s}      s <= t
//   Vnew      = T' (V - diag(e^G) K S)           (S is dk x dv, the state entering the chunk)
//   O         = scale (diag(e^G) Q S + Aqk Vnew)
//   S'        = e^{G_{C-1}} S + K^T diag(e^{G_{C-1} - G}) Vnew
// Only differences G_t - G_s with s <= t are exponentiated, so nothing overflows.
//
// gdn_chunk_prep  -- one workgroup per (b, h, chunk), all chunks in parallel: G by a wave
//   scan, K K^T and Q K^T on v_mfma_f32_32x32x16_f16 (the all-zero upper tile skipped), the
//   exact (I + A)^-1 by 16x16 blocks in fp32.  T' (fp16 hi + lo), Aqk and the per-token factors
//   go to the workspace in the operand layouts the carry loads.
// gdn_chunk_carry -- one workgroup per (b, h, 16 or 32 state columns), sequential over chunks.
//   V and K S meet before T' is applied, so neither T' V nor T' K ever exists in memory: per
//   chunk and head the prep leaves 19 KiB, which the carry reads besides q, k and v's rows
//   (with W = T' diag(e^G) K and U = T' V formed by the prep it was 57 KiB each way: 372 MB per
//   call at 32 heads, T = 4096, against 106 MB of inputs and outputs).
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace tsa {
namespace {

constexpr int kC = 64;     // chunk
constexpr int kD = 128;    // dk = dv
constexpr int kThreads = 256;
constexpr int kCarryThreads = 512;
constexpr int kAbortWgs = 4;  // carry workgroups per head beside the prep (32 columns each)

// Workspace per (b, h, chunk).  T' and Aqk are in operand order: slot (w, ks), lane (g, c) holds
// row 16 w + c, columns 32 ks + 8 g .. + 7 in 16 bytes; the slots (0, 1) and (1, 1) lie above the
// diagonal and are left out.
constexpr int kTSlots = 6;
__device__ __forceinline__ int op_slot(int w, int ks) { return w < 2 ? w : 2 * w - 2 + ks; }
constexpr int kWsT = 0;                            // fp16 T' hi
constexpr int kWsTlo = kWsT + kTSlots * 1024;      // fp16 T' - hi
constexpr int kWsAqk = kWsTlo + kTSlots * 1024;    // fp16 Aqk
// fp32 [64] e^{G_t} qn_t, [64] e^{G_t} kn_t, [64] e^{G_63 - G_t} kn_t, [64] e^{G_63}, where qn_t,
// kn_t are the l2-norm factors of the fused entry point's raw q / k rows (1 otherwise)
constexpr int kWsG = kWsAqk + kTSlots * 1024;
// The chunk's K and Q rows as fp16, written once per QK head (by the V-head of the same number, whose
// slot holds them): K as rows, Q in operand order (slot (w, kk), lane (g, c): token 16 w + c, dk
// 32 kk + 8 g .. + 7), with fp32 I/O then K - fp16(K).  In the inputs a head's rows lie Hq * 256
// bytes apart: with Hq a multiple of 16 they share one L2 channel, and the 8 carry workgroups of
// a head wait for it (T = 4096, 32 heads: 112 us a call with 16 QK heads, 96 us with 11).
constexpr int kWsK = kWsG + kC * 16;
constexpr int kWsQ = kWsK + kC * kD * 2;
constexpr int kWsKlo = kWsQ + kC * kD * 2;
constexpr int kWsUsed = kWsKlo;                  // 52224 B
constexpr int kWsUsedF32 = kWsKlo + kC * kD * 2; // 68608 B
// Bytes from one chunk's workspace to the next: what callers have sized their buffers by
// (tsa_gdn_chunked_workspace_bytes) and what decides whether the no-allocation scratch holds a
// call, so it stays though a chunk now uses less.
constexpr int kWsChunk = 58368;
constexpr int kWsChunkF32 = 107520;
static_assert(kWsUsed <= kWsChunk && kWsUsedF32 <= kWsChunkF32, "a chunk's workspace fits its slot");
template <bool kF32> constexpr int ws_chunk() { return kF32 ? kWsChunkF32 : kWsChunk; }

// Ready flags, after all chunk workspaces: one word per (b, h, chunk), then an abort word per
// carry workgroup.  A call that runs the prep beside the carry first clears them with a small
// kernel on the caller's stream (gdn_flags_clear, a kernel rather than a memset so that a
// captured graph replays it correctly), so whatever the workspace held before, no flag reads
// as set before the prep sets it in this call.  A call that runs them in order writes and
// reads no flags (both kernels get a null flag pointer: the kernel boundary orders the prep's
// stores before the carry), and the carry zeroes the abort words itself.  Beside the carry
// the prep writes 1 there once the chunk's workspace is in memory; the carry's waves wait
// for it before loading the chunk's workspace.
// A wait gives up after a limit on the 100 MHz real-time counter (2 ms; the environment
// variable TSA_GDN_CARRY_WAIT_US sets it in microseconds, 0 = give up whenever a chunk is
// not ready at the first look, which is how the tests exercise the path).  When the prep
// runs beside the carry, a workgroup that gave up leaves its state columns untouched and
// writes 1 to its abort word; a second launch of the carry, ordered after the prep on the
// caller's stream, runs exactly the workgroups whose abort word is 1 and exits at once in the
// others.  Waits time out when the two kernels do not run at the same time: a profiler or a
// runtime setting that serialises dispatches, or a device busy with other work.  The abort
// words stay in the workspace after the call (tsa_gdn_chunked_redo_count reads them).  A
// wait that times out where no second launch follows poisons the state with NaN.

// Wait limit of the second carry launch (1 s); it runs after the prep, so its flags are
// normally all set.
constexpr unsigned kRetryWaitTicks = 100000000u;

// Carry launch modes.
constexpr int kCarryInOrder = 0;  // after the prep on one stream: waits never block
constexpr int kCarryBeside = 1;   // beside the prep: a timed-out workgroup aborts
constexpr int kCarryRetry = 2;    // after the prep: only the first launch's aborted workgroups run

// Sequence split (few heads, many chunks): T is cut into nseg segments of seg_len chunks (the
// last takes the rest).  The state update is linear in the state and in V, so the state
// after a segment is an affine map of the state E entering it, S_out = Phi E + Z, where Z is
// the segment's chain run from S = 0 and Phi its chain run from S = I with V = 0; and a
// chunk's output, O = A S + B, is then O = O_Z + M E, where O_Z is the output of the Z chain
// and M = A Phi_<c the output of the Phi chain (V = 0 makes B vanish).  Three launches after
// the prep:
//   maps    -- segment 0's chain from the caller's state (its outputs, and its end state as
//              segment 1's entry), and, side by side, the Z and Phi chains of segments
//              1 .. nseg-1 with their outputs O_Z and M (fp32, to the workspace);
//   combine (gdn_seg_combine) -- E[s+1] = Phi_s E[s] + Z_s for s = 1 .. nseg-1, the last
//              one the call's final state;
//   fixup   (gdn_seg_fixup) -- O = O_Z + M E for every chunk of segments 1 .. nseg-1, all
//              chunks in parallel.
// The serial depth drops from nch chunk steps to seg_len chunk steps + nseg - 1 combine
// steps.  Per (b, h, segment) the workspace holds three [128 columns][128] fp32 slots
// (entry E, Z, Phi), and per (b, h) the O_Z and M rows of the tokens after segment 0.
constexpr int kJobPlain = 0, kJobMaps = 1;
constexpr int kSegSlots = 3, kSegEntry = 0, kSegZ = 1, kSegPhi = 2;
constexpr size_t kSegSlotFloats = (size_t)kD * kD;
struct CarryJob {
    int phase = kJobPlain;
    int nseg = 1, seg_len = 0;
    int Tr = 0;            // tokens after segment 0: rows of oz / om per (b, h)
    float* seg = nullptr;  // [B*Hv][nseg][kSegSlots][kD][kD]
    float* oz = nullptr;   // [B*Hv][Tr][kD]: O_Z, the Z chains' outputs
    float* om = nullptr;   // [B*Hv][Tr][kD]: M, the Phi chains' outputs
};

// 16-B chunk swizzle for [rows][128] fp16 LDS tiles (same argument as attn_fwd.hip): 16
// consecutive rows at one chunk, and 4 aligned rows x 2 chunks, are bank-conflict free.
__device__ __forceinline__ int swz(int r) {
    return 2 * (r & 3) + ((r >> 2) & 1) + 8 * ((r >> 3) & 1);
}
__device__ __forceinline__ int tile_off(int r, int c /*16-B chunk*/) {
    return r * kD + ((c ^ swz(r)) << 3);
}
// Transposed read of a [rows][128] tile: within each 16-lane group the result lane holds
// column col0 + lane%16 for rows row0 .. row0+3 (this lane supplies row0 + (l%16)/4).
__device__ __forceinline__ half4_t tile_read_tr(const half_t* tile, int row0, int col0) {
    const int i16 = threadIdx.x & 15;
    const int r = row0 + (i16 >> 2);
    const int col = col0 + 4 * (i16 & 3);
    return lds_read_tr16(tile + tile_off(r, col >> 3) + (col & 7));
}

// Orders this wave's LDS writes before its later LDS reads of other lanes' data.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ half8_t cat8(const half4_t& a, const half4_t& b) {
    return half8_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// Device-scope stores of the workspace (sc1): written through to the device's coherence
// point, so a carry beside the prep, whose loads of them are device-scope too, sees them from any
// XCD as soon as this wave's vmcnt has drained -- no L2 write-back or invalidate needed
// (both measured far too slow to issue once per workgroup or chunk).
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store_dev(unsigned char* p, const uint4& v) {
    const u32x4_t x = {v.x, v.y, v.z, v.w};
    // s_nop 1: a store of more than 8 bytes may still read its data registers in the next
    // cycle, and the compiler does not see into this asm to keep them unchanged that long
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(x) : "memory");
}
__device__ __forceinline__ void store_dev8(unsigned char* p, const uint2& v) {
    const u32x2_t x = {v.x, v.y};
    asm volatile("global_store_dwordx2 %0, %1, off sc1" ::"v"(p), "v"(x) : "memory");
}
__device__ __forceinline__ void store_dev(float* p, float v) {
    asm volatile("global_store_dword %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
}

// x as a value in a register.  The two halves of a split must come from the same fp32 value: left
// alone, the compiler folds a product into the high half's conversion (one rounding) but not
// into the low half's subtraction, and a product near a tie loses half an fp16 ulp.
__device__ __forceinline__ float rounded(float x) {
    asm volatile("" : "+v"(x));
    return x;
}

// 8 consecutive q / k / v elements as 8 fp16 values (one uint4), from fp16 or fp32 memory:
// fp32 inputs are converted in registers.
__device__ __forceinline__ uint4 load8h(const half_t* p) { return *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ uint4 load8h(const float* p) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    const half8_t h = {(half_t)a.x, (half_t)a.y, (half_t)a.z, (half_t)a.w,
                       (half_t)b.x, (half_t)b.y, (half_t)b.z, (half_t)b.w};
    return __builtin_bit_cast(uint4, h);
}
// The same 8 elements as an exact pair of fp16 halves: hi = fp16(x), lo = fp16(x - hi).
__device__ __forceinline__ void load8hl(const float* p, uint4& hi, uint4& lo) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    half8_t h, l;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        h[e] = (half_t)x[e];
        l[e] = (half_t)(x[e] - (float)h[e]);
    }
    hi = __builtin_bit_cast(uint4, h);
    lo = __builtin_bit_cast(uint4, l);
}
__device__ __forceinline__ void load8hl(const half_t* p, uint4& hi, uint4&) { hi = load8h(p); }

// ----------------------------------------------------------------------------------
// Prep
// ----------------------------------------------------------------------------------
// Packed storage of the ten lower-triangular 16x16 fp32 blocks of a 64 x 64 matrix (A, Tm):
// block (i, j), j <= i, at (i(i+1)/2 + j) * 256 floats, element (r, c) of a block at
// 16 r + 4 ((c/4) ^ (r/4 % 4)) + c % 4.  The XOR of 16-byte chunks makes the MFMA operand
// reads of the block solve (16 rows x 4 columns, 4 rows x 16 columns) hit 64 distinct
// banks, and keeps 4 consecutive columns in one 16-byte chunk.
__device__ __forceinline__ int tri_off(int row, int col) {
    const int i = row >> 4, j = col >> 4, r = row & 15, c = col & 15;
    return (((i * (i + 1)) >> 1) + j) * 256 + r * 16 + ((((c >> 2) ^ (r >> 2)) & 3) << 2) + (c & 3);
}

// A and Tm take the places of the Q and K rows once K K^T and Q K^T are done.
struct PrepLds {
    union {
        half_t K[kC * kD];     // K rows, swizzled
        float Tm[10 * 256];    // (I + A)^-1, packed blocks
    };
    union {
        half_t Q[kC * kD];     // Q rows, swizzled
        float A[10 * 256];     // strictly lower A, packed blocks
    };
    float G[kC];
    float bt[kC];
    float kn[kC];  // l2-norm factors 1 / max(||k_t||, eps), 1 / max(||q_t||, eps) (fused only)
    float qn[kC];
};

// kFused: q / k are the raw rows (normalised here: the factors scale A, Aqk and the per-token
// factors, so the carry takes the raw K / Q rows), and g_log / beta are computed from the raw
// projections a / b (gate arguments).
// TIO: the q / k element type.
// With fp32 I/O K K^T takes K as hi + lo (hi hi + hi lo + lo hi): the carry's K S does, and an A of
// rounded rows beside it would be its state error (1.0e-4 instead of 1e-5 on a slow gate, T = 2048).
template <typename TIO> constexpr int prep_wgs_per_cu() { return std::is_same<TIO, float>::value ? 3 : 4; }
template <bool kFused, typename TIO>
__global__ void __launch_bounds__(kThreads, prep_wgs_per_cu<TIO>())
gdn_chunk_prep(const TIO* __restrict__ q, const TIO* __restrict__ k, const float* __restrict__ g_log,
               const float* __restrict__ beta, GdnRawGates gates, unsigned char* __restrict__ ws,
               unsigned* __restrict__ flags, int T, int Hq, int Hv, int nch, int BHv, GdnStrides st) {
    __shared__ __align__(16) PrepLds sm;
    __shared__ __align__(16) half_t klo_lds[std::is_same<TIO, float>::value ? kC * kD : 8];  // low halves of the K rows
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hi = lane >> 5;
    // chunk-major: workgroups are dispatched in the order the carry consumes chunks, and
    // (b, h, chunk) lands on the XCD of the head's carry workgroups when BHv % 8 == 0
    const int ch = blockIdx.x / BHv;
    const int bh = blockIdx.x % BHv;
    const int b = bh / Hv, h = bh % Hv, hq = h % Hq;
    const int t0 = ch * kC;
    constexpr bool kF32 = std::is_same<TIO, float>::value;
    unsigned char* wsc = ws + ((size_t)bh * nch + ch) * ws_chunk<kF32>();
    const int mt = wave >> 1, nt = wave & 1;  // this wave's 32x32 tile of K K^T / Q K^T

    // ---- 1. K and Q rows to LDS.  Every global load of the phase is issued first (wave 0's gate
    // inputs, K, Q), from row-clamped addresses, and rows past T are zeroed where the values are
    // consumed: a branch around a load makes the compiler wait for every load in flight where the
    // paths join.  A row is 16 lanes of 16 bytes: loading Q in the shape of its MFMA operand (32
    // rows x 32 bytes an instruction) cost 128 cycles of the CU's load path each instead of 20 ----
    const int lastt = T - 1;
    float gx = 0.f, gy = 0.f;  // wave 0: the gate inputs of token t0 + lane
    if (wave == 0) {
        const size_t bt = (size_t)b * T + min(t0 + lane, lastt);
        gx = kFused ? gates.a[bt * Hv + h] : g_log[bt * Hv + h];
        gy = kFused ? gates.b[bt * Hv + h] : beta[bt * Hv + h];
    }
    uint4 kreg[4], qreg[4], klo[4];
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int id = it * kThreads + tid;
        const int t = min(t0 + (id >> 4), lastt);
        load8hl(k + b * st.k.b + t * st.k.t + hq * st.k.h + (id & 15) * 8, kreg[it], klo[it]);
        qreg[it] = load8h(q + b * st.q.b + t * st.q.t + hq * st.q.h + (id & 15) * 8);
    }
    const bool copies = h < Hq;  // this workgroup leaves its QK head's rows to the carry
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int id = it * kThreads + tid;
        const int r = id >> 4, c = id & 15;
        const bool past = t0 + r > lastt;
        const uint4 kv = past ? make_uint4(0, 0, 0, 0) : kreg[it], qv = past ? make_uint4(0, 0, 0, 0) : qreg[it];
        const uint4 kl = past ? make_uint4(0, 0, 0, 0) : klo[it];
        *reinterpret_cast<uint4*>(sm.K + tile_off(r, c)) = kv;
        *reinterpret_cast<uint4*>(sm.Q + tile_off(r, c)) = qv;
        if (kF32) *reinterpret_cast<uint4*>(klo_lds + tile_off(r, c)) = kl;
        if (copies) {
            store_dev(wsc + kWsK + (size_t)id * 16, kv);
            if (kF32) store_dev(wsc + kWsKlo + (size_t)id * 16, kl);
        }
        if (kFused) {  // the row's 16 threads are 16 consecutive lanes of one wave
            const half8_t k8 = __builtin_bit_cast(half8_t, kv), q8 = __builtin_bit_cast(half8_t, qv);
            float sk = 0.f, sq = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sk = fmaf((float)k8[e], (float)k8[e], sk);
                sq = fmaf((float)q8[e], (float)q8[e], sq);
            }
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) {
                sk += __shfl_xor(sk, off);
                sq += __shfl_xor(sq, off);
            }
            if (c == 0) {
                sm.kn[r] = 1.f / fmaxf(sqrtf(sk), gates.eps);
                sm.qn[r] = 1.f / fmaxf(sqrtf(sq), gates.eps);
            }
        }
    }
    if (wave == 0) {
        float x = 0.f, be = 0.f;
        if (t0 + lane <= lastt) {
            if (kFused) {
                x = gdn_softplus(gx + gates.dt_bias[h]) * gates.A[h];
                be = gdn_sigmoid(gy);
            } else {
                x = gx;
                be = gy;
            }
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {  // inclusive prefix sum over the chunk
            const float y = __shfl_up(x, off);
            if (lane >= off) x += y;
        }
        sm.G[lane] = x;
        sm.bt[lane] = be;
    }
    lds_barrier();
    if (copies) {  // Q in operand order
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int id = it * kThreads + tid, sl = id >> 6, l = id & 63;
            store_dev(wsc + kWsQ + (size_t)id * 16,
                      *reinterpret_cast<const uint4*>(sm.Q + tile_off(16 * (sl >> 2) + (l & 15), 4 * (sl & 3) + (l >> 4))));
        }
    }

    // ---- 2. K K^T and Q K^T, transposed (a lane holds token t = 32 mt + lane % 32 and keys
    // s = 32 nt + 8 q + 4 hi + 0..3 in registers 4q..4q+3): A goes to LDS in 16-byte pieces, Aqk
    // straight to the workspace in 8-byte pieces of the carry's operand order ----
    const bool upper = mt == 0 && nt == 1;
    const int t = 32 * mt + (lane & 31), rs = 32 * nt + (lane & 31);
    float16_t kk = {}, qk = {};
    if (!upper) {
#pragma unroll
        for (int s = 0; s < kD / 16; ++s) {
            const int c = 2 * s + hi;
            const half8_t at = *reinterpret_cast<const half8_t*>(sm.K + tile_off(t, c));
            const half8_t bs = *reinterpret_cast<const half8_t*>(sm.K + tile_off(rs, c));
            const half8_t qa = *reinterpret_cast<const half8_t*>(sm.Q + tile_off(t, c));
            kk = mfma32(bs, at, kk);
            if (kF32) {
                kk = mfma32(*reinterpret_cast<const half8_t*>(klo_lds + tile_off(rs, c)), at, kk);
                kk = mfma32(bs, *reinterpret_cast<const half8_t*>(klo_lds + tile_off(t, c)), kk);
            }
            qk = mfma32(bs, qa, qk);
        }
    }
    lds_barrier();  // every wave's Q reads done: A goes over them
    if (upper) {
        // every (t < 32, s >= 32) entry is above the diagonal (the carry reads no Aqk there);
        // this wave writes the per-token factors instead
        const float x = sm.G[lane], xc = sm.G[kC - 1];
        const float ex = __expf(x);
        const float kn = kFused ? sm.kn[lane] : 1.f, qn = kFused ? sm.qn[lane] : 1.f;
        float* wg = reinterpret_cast<float*>(wsc + kWsG);
        store_dev(wg + lane, ex * qn);
        store_dev(wg + kC + lane, ex * kn);
        store_dev(wg + 2 * kC + lane, __expf(xc - x) * kn);
        store_dev(wg + 3 * kC + lane, __expf(xc));
    } else {
        const float Gt = sm.G[t];
        float bt = sm.bt[t], qf = 1.f;
        if (kFused) {
            bt *= sm.kn[t];
            qf = sm.qn[t];
        }
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
            const int s0 = 32 * nt + 8 * qd + 4 * hi;
            const float4 g4 = *reinterpret_cast<const float4*>(sm.G + s0);
            const float gs[4] = {g4.x, g4.y, g4.z, g4.w};
            float ks[4] = {1.f, 1.f, 1.f, 1.f};
            if (kFused) {
                const float4 k4 = *reinterpret_cast<const float4*>(sm.kn + s0);
                ks[0] = k4.x; ks[1] = k4.y; ks[2] = k4.z; ks[3] = k4.w;
            }
            float av[4];
            half4_t qv;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float dec = s0 + e <= t ? __expf(Gt - gs[e]) * ks[e] : 0.f;
                av[e] = s0 + e < t ? bt * kk[4 * qd + e] * dec : 0.f;
                qv[e] = (half_t)(qk[4 * qd + e] * (dec * qf));
            }
            // blocks above the diagonal (t / 16 < s / 16) are not stored
            if (mt != nt || qd < 2 || (lane & 16))
                *reinterpret_cast<float4*>(sm.A + tri_off(t, s0)) = make_float4(av[0], av[1], av[2], av[3]);
            store_dev8(wsc + kWsAqk + (size_t)((op_slot(t >> 4, nt) * 64 + qd * 16 + (t & 15)) * 16 + 8 * hi),
                       __builtin_bit_cast(uint2, qv));
        }
    }
    lds_barrier();

    // ---- 3. Tm = (I + A)^-1 ----
    if (wave == 0) {  // the four 16x16 diagonal blocks, one column per lane
        const int bi = lane >> 4, cj = lane & 15;
        float x[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) x[t] = t == cj ? 1.f : 0.f;
        // row t of the block in 16-byte pieces; every row's earlier columns are known when it
        // is reached, and its products go to one running sum (s ascending)
#pragma unroll
        for (int t = 1; t < 16; ++t) {
            float a[16];
#pragma unroll
            for (int s4 = 0; s4 < 16; s4 += 4) {
                if (s4 >= t) break;
                const float4 v = *reinterpret_cast<const float4*>(sm.A + tri_off(16 * bi + t, 16 * bi + s4));
                a[s4] = v.x; a[s4 + 1] = v.y; a[s4 + 2] = v.z; a[s4 + 3] = v.w;
            }
            float acc = x[t];
#pragma unroll
            for (int s = 0; s < t; ++s) acc = fmaf(-a[s], x[s], acc);
            x[t] = acc;
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) sm.Tm[tri_off(16 * bi + t, 16 * bi + cj)] = x[t];
    }
    lds_barrier();
    if (wave < 3) {  // block column j = wave: T_ij = -T_ii X, X = sum_{k=j}^{i-1} A_ik T_kj, i > j
        // 16x16x16 fp32 block products on v_mfma_f32_16x16x4_f32 (lane l: A[l%16][l/16],
        // B[l/16][l%16], D[4*(l/16) + r][l%16]); the diagonal blocks hold zeros above the
        // diagonal, so no masking is needed.  X stays in registers: register s of lane l
        // holds X[4*(l/16) + s][l%16], which is the B operand of k-step s when the A operand
        // supplies column 4*(l/16) + s of T_ii.
        const int j = wave, r16 = lane & 15, k4 = lane >> 4;
        for (int i = j + 1; i < 4; ++i) {
            float4_t x = {};
            for (int kb = j; kb < i; ++kb)
#pragma unroll
                for (int s4 = 0; s4 < 4; ++s4)
                    x = mfma16f32(sm.A[tri_off(16 * i + r16, 16 * kb + 4 * s4 + k4)],
                                  sm.Tm[tri_off(16 * kb + 4 * s4 + k4, 16 * j + r16)], x);
            float4_t t = {};
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4)
                t = mfma16f32(sm.Tm[tri_off(16 * i + r16, 16 * i + 4 * k4 + s4)], x[s4], t);
#pragma unroll
            for (int r = 0; r < 4; ++r) sm.Tm[tri_off(16 * i + 4 * k4 + r, 16 * j + r16)] = -t[r];
            wave_lds_sync();
        }
    }
    lds_barrier();

    // ---- 4. T' = Tm diag(beta) as an exact pair of fp16 halves, in the carry's operand order
    // (slot (w, ks), lane (g, c): T'[16 w + c][32 ks + 8 g .. + 7]) ----
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int id = it * kThreads + tid;
        if (id >= kTSlots * 64) break;
        const int sl = id >> 6, l = id & 63;
        const int w = sl < 2 ? sl : 2 + ((sl - 2) >> 1), ks = sl < 2 ? 0 : (sl - 2) & 1;
        const int t = 16 * w + (l & 15), s0 = 32 * ks + 8 * (l >> 4);
        // a block above the diagonal is zero; the read goes to a stored block instead
        const int base = tri_off(t, 16 * min(s0 >> 4, t >> 4) + (s0 & 8));
        const float4 t0v = *reinterpret_cast<const float4*>(&sm.Tm[base]);
        const float4 t1v = *reinterpret_cast<const float4*>(&sm.Tm[base ^ 4]);
        const float4 b0v = *reinterpret_cast<const float4*>(sm.bt + s0);
        const float4 b1v = *reinterpret_cast<const float4*>(sm.bt + s0 + 4);
        const float tv[8] = {t0v.x, t0v.y, t0v.z, t0v.w, t1v.x, t1v.y, t1v.z, t1v.w};
        const float bv[8] = {b0v.x, b0v.y, b0v.z, b0v.w, b1v.x, b1v.y, b1v.z, b1v.w};
        half8_t th, tl;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float y = rounded(s0 + e <= t ? tv[e] * bv[e] : 0.f);
            th[e] = (half_t)y;
            tl[e] = (half_t)(y - (float)th[e]);
        }
        const size_t o = (size_t)id * 16;
        store_dev(wsc + kWsT + o, __builtin_bit_cast(uint4, th));
        store_dev(wsc + kWsTlo + o, __builtin_bit_cast(uint4, tl));
    }

    // ---- 5. publish (beside the carry only): every wave's device-scope stores complete, then
    // the chunk's flag.  In order the kernel boundary orders the stores before the carry, so
    // the workgroup ends without waiting for them ----
    if (flags) {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        __builtin_amdgcn_s_barrier();
        if (tid == 0)
            __hip_atomic_store(flags + (size_t)bh * nch + ch, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ----------------------------------------------------------------------------------
// Carry
// ----------------------------------------------------------------------------------
// One workgroup of 8 waves per (b, h, 16 NC state columns), sequential over chunks.
//
// Chain waves 0-3 run the loop-carried part.  Wave w owns tokens 16 w .. + 15 of the chunk (rows
// of K S and T' R) and state rows dk 32 w .. + 31 (fp32 accumulators) for all of the workgroup's
// columns, so it reads a quarter of each operand; what the waves exchange goes through LDS in
// operand order (16-byte lane-linear reads).  Per chunk, a barrier after each:
//   1  X = K S, R = V - e^G X as fp16 hi + lo -> LDS
//   2  Vnew = T' R (hi hi + lo hi + hi lo); Vnew and Vnew e^{G_63 - G} (hi + lo) -> LDS
//   3  S = e^{G_63} S + K^T (hi + lo); S -> LDS as fp16
// Helper waves 4-7 do everything that touches memory, in the same three intervals: wave w's
// output tokens are 16 w .. + 15.
//   1  the next chunk's K, V and factors from registers to LDS
//   2  its T'; (Q S)^T for the wave's tokens
//   3  O = e^G Q S + Aqk Vnew, stored
// Every operand is loaded into registers two or three chunks before its use and its registers are reloaded as soon as they are free, a few loads in each interval: a wave that
// issues loads stalls at issue while the CU's 64 B/clk load path is busy (~50 KB per chunk, 800
// cycles), which in the chain waves cost 1.6 us per chunk instead of the chain's own time.
template <typename TIO, int NC>
struct CarrySlot {                      // a chunk's operands of the chain waves
    static constexpr bool kF32 = std::is_same<TIO, float>::value;
    half_t K[(kF32 ? 2 : 1) * kC * kD]; // K rows, swizzled (fp32 I/O: then their low halves)
    uint4 T[kTSlots * 2 * 64];          // T' hi, lo in operand order
    TIO V[kC * 16 * NC];                // [token][column index 4 NC (i / 4) ...] as in memory
    float G[4 * kC];                    // the per-token factors
};
template <typename TIO, int NC>
struct CarryLds {
    static constexpr bool kF32 = std::is_same<TIO, float>::value;
    CarrySlot<TIO, NC> c[2];
    uint4 S[kF32 ? 2 : 1][NC][4][64];   // state operand, k-step, lane (fp32 I/O: hi, lo)
    uint4 R[2][NC][2][64];              // R hi, lo
    uint4 Rb[2][NC][2][64];             // 2^-16 R hi, lo where |R| > kMaxHalf (written only then)
    union {
        unsigned char big[4];           // per chain wave: its rows of Rb hold this chunk's values
        unsigned bigs;
    };
    uint4 V[3][NC][2][64];              // Vnew e^{G_63 - G} hi, lo; Vnew
    int err[4];                         // per helper wave: a ready wait timed out
};

__device__ __forceinline__ uint4 bload4(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
// workspace loads beside the prep are device-scope (sc1), the counterpart of its stores
template <bool kDev>
__device__ __forceinline__ uint4 bload4w(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kDev ? 16 : 0));
}
template <bool kDev>
__device__ __forceinline__ float bload1w(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, kDev ? 16 : 0));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
}

// 4 fp32 values as 4 fp16 highs and 4 fp16 lows.
__device__ __forceinline__ void split4(const float4_t& x, uint2& hi, uint2& lo) {
    half4_t h, l;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float y = rounded(x[r]);
        h[r] = (half_t)y;
        l[r] = (half_t)(y - (float)h[r]);
    }
    hi = __builtin_bit_cast(uint2, h);
    lo = __builtin_bit_cast(uint2, l);
}

// R = V - e^G K S may lie beyond the fp16 range where Vnew = T' R does not (beta, a factor of T', is
// small).  Such entries go to T' as 2^-16 R in a pair of their own, and 0 in R's place.
constexpr float kMaxHalf = 65504.f;

// Keeps the loads after it behind the products that make x.  Every reload must stay behind the
// last use of what it replaces: with a use left below it the compiler takes other registers for
// the new value and copies them at the loop's end, waiting for a load just issued.
__device__ __forceinline__ void pin(float4_t& x) { asm volatile("" : "+v"(x)::"memory"); }

// TIO: the q / k / v / out element type.  NC: 16-column tiles of the workgroup.  kFlags: the
// call runs beside the prep (or is its second launch) and waits on the chunks' ready flags.
// job: the whole sequence (kJobPlain), or the maps launch of the sequence split (segments of the
// workgroup's unit, its start state and where its end state goes are derived below).
// One workgroup per CU: two waves per SIMD, one of each role.
// kWide: V and the output are addressed in 64 bits a lane instead of by descriptors of a chunk's 64
// rows, for rows of 2^31 / 64 bytes and more (65 536 heads in fp32, 131 072 in fp16).
template <typename TIO, int NC, bool kFlags, bool kWide = false>
__global__ void __launch_bounds__(kCarryThreads, 2)
gdn_chunk_carry(const TIO* __restrict__ v, const unsigned char* __restrict__ ws, const unsigned* __restrict__ flags,
                unsigned* __restrict__ aborts, int mode, unsigned wait_ticks, const float* state_in, float* state,
                TIO* __restrict__ out, int T, int Hq, int Hv, int nch_all, int BHv, float scale, CarryJob job,
                RowStride vs) {
    constexpr bool kF32 = std::is_same<TIO, float>::value;
    constexpr int kWgs = kD / (16 * NC);  // workgroups per head
    __shared__ __align__(16) CarryLds<TIO, NC> sm;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: role branches are scalar
    const bool chain = wave < 4;
    const int w = wave & 3;
    const int g = lane >> 4, c = lane & 15;
    // Workgroups go round robin over the 8 XCDs.  A head's column parts share an XCD, whose L2 then
    // fetches the head's operands once: the heads are padded to a multiple of 8 and the padding's
    // workgroups end here.  (Not in a maps launch, whose units fill the device: there a head's
    // share of one XCD's CUs would be too many.)
    const int BHp = job.phase == kJobPlain ? (BHv + 7) & ~7 : BHv;
    const int unit = blockIdx.x / (kWgs * BHp);
    const int part = (blockIdx.x / BHp) % kWgs;
    const int bh = blockIdx.x % BHp;
    if (bh >= BHv) return;
    const int wg = part * BHv + bh;  // its abort word (the launches that use one have one unit)
    if (kFlags && mode == kCarryRetry &&
        __builtin_amdgcn_readfirstlane(__hip_atomic_load(aborts + wg, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT)) == 0u)
        return;  // this workgroup finished in the launch beside the prep
    const int b = bh / Hv, h = bh % Hv, hq = h % Hq;

    // This workgroup's chunks [c0, c0 + nch), where its state starts (src: loaded; else zero,
    // or the identity for a transition map), where it ends (dst), where its outputs go (out,
    // or a map's fp32 rows in the workspace), and the V scale (0 for a transition map).
    int seg = 0, c0 = 0, nch = nch_all;
    bool ident = false;
    float us = 1.f;
    const float* src = state_in;
    float* dst = state;
    float* obuf = nullptr;  // a map's fp32 output rows (from segment 1's first token), or out
    // this head's slots (no slots in the plain job)
    float* segh = job.seg ? job.seg + (size_t)bh * job.nseg * kSegSlots * kSegSlotFloats : nullptr;
    auto slot = [&](int sg, int which) { return segh + ((size_t)sg * kSegSlots + which) * kSegSlotFloats; };
    if (job.phase == kJobMaps) {
        if (unit == 0) {            // segment 0 from the caller's state; its end enters segment 1
            dst = slot(1, kSegEntry);
        } else {                    // Z or Phi of segment 1 + (unit - 1) / 2
            seg = 1 + (unit - 1) / 2;
            const bool phi = ((unit - 1) & 1) != 0;
            src = nullptr;
            ident = phi;
            us = phi ? 0.f : 1.f;
            dst = slot(seg, phi ? kSegPhi : kSegZ);
            obuf = (phi ? job.om : job.oz) + ((size_t)bh * job.Tr + (size_t)(seg - 1) * job.seg_len * kC) * kD;
        }
    }
    if (job.phase != kJobPlain) {
        c0 = seg * job.seg_len;
        nch = seg == job.nseg - 1 ? nch_all - c0 : job.seg_len;
    }
    const int Tloc = T - c0 * kC;  // tokens from this workgroup's first chunk to the end of the sequence

    // This lane's columns: with two tiles the columns interleave (tile ct, index i is column
    // 8 (i / 4) + 4 ct + i % 4), so that the transposed output gives a lane 8 consecutive ones.
    const int col0 = part * 16 * NC;
    auto col = [&](int ct, int i) { return col0 + (NC == 1 ? i : 8 * (i >> 2) + 4 * ct + (i & 3)); };
    const int nks = w < 2 ? 1 : 2;  // T' and Aqk key steps on or below the diagonal, from slot ts
    const int ts = w < 2 ? w : 2 * w - 2;

    if (chain) {
        // state layout [b*Hv + h][column][dk]: rows dk 32 w + 16 m + 4 g + 0..3
        float4_t S[NC][2];
#pragma unroll
        for (int ct = 0; ct < NC; ++ct)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int d0 = 32 * w + 16 * m + 4 * g;
                if (src) {
                    const float4 x = *reinterpret_cast<const float4*>(
                        (src == state_in ? state_in + (size_t)bh * kSegSlotFloats : src) + (size_t)col(ct, c) * kD + d0);
                    S[ct][m] = float4_t{x.x, x.y, x.z, x.w};
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) S[ct][m][r] = ident && d0 + r == col(ct, c) ? 1.f : 0.f;
                }
            }
        // where this lane's 4 consecutive rows of a D tile go in the operand of the next product:
        // row 16 m' + 4 g + r of a 32-row k-step is slot (g' = 2 m' + g / 2, 4 (g % 2) + r)
        auto put = [&](uint4* op, int m, const uint2& x) {
            reinterpret_cast<uint2*>(op)[2 * ((2 * m + (g >> 1)) * 16 + c) + (g & 1)] = x;
        };
        auto put_state = [&]() {
#pragma unroll
            for (int ct = 0; ct < NC; ++ct)
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    uint2 hi, lo;
                    split4(S[ct][m], hi, lo);
                    put(sm.S[0][ct][w], m, hi);
                    if (kF32) put(sm.S[kF32 ? 1 : 0][ct][w], m, lo);
                }
        };
        auto put_r = [&](uint4 (&R)[2][NC][2][64], int ct, const float4_t& x) {
            uint2 hi, lo;
            split4(x, hi, lo);
            put(R[0][ct][w >> 1], w & 1, hi);
            put(R[1][ct][w >> 1], w & 1, lo);
        };
        auto put_v = [&](int ct, const float4_t& x, const float (&dg)[4]) {
            float4_t vs;
            half4_t vh;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                vs[r] = x[r] * dg[r];
                vh[r] = (half_t)x[r];
            }
            uint2 hi, lo;
            split4(vs, hi, lo);
            put(sm.V[0][ct][w >> 1], w & 1, hi);
            put(sm.V[1][ct][w >> 1], w & 1, lo);
            put(sm.V[2][ct][w >> 1], w & 1, __builtin_bit_cast(uint2, vh));
        };
        // step 1's operands that do not depend on the state, read ahead of the barrier before it
        half8_t kA[4], kAl[4];
        float v[NC][4], ek[4];
        half4_t v4[NC];
        auto ahead = [&](const CarrySlot<TIO, NC>& cs) __attribute__((always_inline)) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                kA[kk] = *reinterpret_cast<const half8_t*>(cs.K + tile_off(16 * w + c, 4 * kk + g));
                if (kF32) kAl[kk] = *reinterpret_cast<const half8_t*>(cs.K + kC * kD + tile_off(16 * w + c, 4 * kk + g));
            }
            // V of tokens 16 w + 4 g + r at this lane's columns (fp16: read transposed, the lane
            // supplying 4 columns of one token)
#pragma unroll
            for (int ct = 0; ct < NC; ++ct)
                if constexpr (kF32) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[ct][r] = cs.V[(16 * w + 4 * g + r) * 16 * NC + col(ct, c) - col0];
                } else {
                    v4[ct] = lds_read_tr16(cs.V + (16 * w + 4 * g + (c >> 2)) * 16 * NC + col(ct, 4 * (c & 3)) - col0);
                }
            const float4 e = *reinterpret_cast<const float4*>(cs.G + kC + 16 * w + 4 * g);
            ek[0] = e.x; ek[1] = e.y; ek[2] = e.z; ek[3] = e.w;
        };
        if (lane == 0) sm.big[w] = 0;
        auto step = [&](const CarrySlot<TIO, NC>& cs, const CarrySlot<TIO, NC>& nx) __attribute__((always_inline)) {
            // ---- 1. X = K S; R = V - e^G X ----
            half8_t Sh[NC][4], Sl[NC][4];
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                for (int ct = 0; ct < NC; ++ct) {
                    Sh[ct][kk] = __builtin_bit_cast(half8_t, sm.S[0][ct][kk][lane]);
                    if (kF32) Sl[ct][kk] = __builtin_bit_cast(half8_t, sm.S[kF32 ? 1 : 0][ct][kk][lane]);
                }
            // T' operands of step 2: their LDS time runs under step 1
            half8_t th[2], tl[2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                th[ks] = __builtin_bit_cast(half8_t, cs.T[(ts + min(ks, nks - 1)) * 64 + lane]);
                tl[ks] = __builtin_bit_cast(half8_t, cs.T[(kTSlots + ts + min(ks, nks - 1)) * 64 + lane]);
            }
            __builtin_amdgcn_sched_barrier(0);
            float4_t R[NC];
            float m = 0.f;
#pragma unroll
            for (int ct = 0; ct < NC; ++ct) {
                float4_t x[2] = {};
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    x[kk & 1] = mfma16(kA[kk], Sh[ct][kk], x[kk & 1]);
                    if (kF32) {
                        x[kk & 1] = mfma16(kA[kk], Sl[ct][kk], x[kk & 1]);
                        x[kk & 1] = mfma16(kAl[kk], Sh[ct][kk], x[kk & 1]);
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) R[ct][r] = fmaf(-ek[r], x[0][r] + x[1][r], us * (kF32 ? v[ct][r] : (float)v4[ct][r]));
                put_r(sm.R, ct, R[ct]);
                m = fmaxf(m, fmaxf(fmaxf(fabsf(R[ct][0]), fabsf(R[ct][1])), fmaxf(fabsf(R[ct][2]), fabsf(R[ct][3]))));
            }
            // Behind the whole step and out of line: a branch between the tiles cost 4 % of a call of
            // 48 heads, T = 4096, this form 1.5 % (113.5 -> 115.0 us; 32 heads 89.9 -> 88.2).
            const bool big = __builtin_amdgcn_ballot_w64(m > kMaxHalf) != 0;
            if (__builtin_expect(big, 0)) {
#pragma unroll
                for (int ct = 0; ct < NC; ++ct) {
                    float4_t y;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const bool out = fabsf(R[ct][r]) > kMaxHalf;
                        y[r] = out ? R[ct][r] * 0x1p-16f : 0.f;
                        if (out) R[ct][r] = 0.f;
                    }
                    put_r(sm.R, ct, R[ct]);
                    put_r(sm.Rb, ct, y);
                }
                if (lane == 0) sm.big[w] = 1;
            }
            lds_barrier();
            // ---- 2. Vnew = T' R ----
            half8_t Rh[NC][2], Rl[NC][2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int ct = 0; ct < NC; ++ct) {
                    Rh[ct][ks] = __builtin_bit_cast(half8_t, sm.R[0][ct][ks][lane]);
                    Rl[ct][ks] = __builtin_bit_cast(half8_t, sm.R[1][ct][ks][lane]);
                }
            const unsigned bigs = sm.bigs;
            // K^T operands and factors of step 3 (and e^{G_63 - G}): under step 2
            half8_t aK[2][2], aKl[2][2];
            const float4 d4 = *reinterpret_cast<const float4*>(cs.G + 2 * kC + 16 * w + 4 * g);
            const float ec = cs.G[3 * kC];
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    aK[m][ks] = cat8(tile_read_tr(cs.K, 32 * ks + 8 * g, 32 * w + 16 * m),
                                     tile_read_tr(cs.K, 32 * ks + 8 * g + 4, 32 * w + 16 * m));
                    if (kF32)
                        aKl[m][ks] = cat8(tile_read_tr(cs.K + kC * kD, 32 * ks + 8 * g, 32 * w + 16 * m),
                                          tile_read_tr(cs.K + kC * kD, 32 * ks + 8 * g + 4, 32 * w + 16 * m));
                }
            __builtin_amdgcn_sched_barrier(0);
            const float dg[4] = {d4.x, d4.y, d4.z, d4.w};
            float4_t V[NC];
#pragma unroll
            for (int ct = 0; ct < NC; ++ct) {
                float4_t vn[3] = {};
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    if (ks >= nks) break;  // uniform
                    vn[0] = mfma16(th[ks], Rh[ct][ks], vn[0]);
                    vn[1] = mfma16(tl[ks], Rh[ct][ks], vn[1]);
                    vn[2] = mfma16(th[ks], Rl[ct][ks], vn[2]);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) V[ct][r] = vn[0][r] + (vn[1][r] + vn[2][r]);
                put_v(ct, V[ct], dg);
            }
            if (__builtin_expect(__builtin_amdgcn_readfirstlane(bigs) != 0, 0)) {
#pragma unroll
                for (int ct = 0; ct < NC; ++ct) {
                    float4_t y = {};
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks) {
                        if (ks >= nks) break;
                        // this lane's 8 rows of the k-step are those of wave 2 ks + g / 2
                        const bool in = (bigs >> (8 * (2 * ks + (g >> 1)))) & 1;
                        const half8_t h = in ? __builtin_bit_cast(half8_t, sm.Rb[0][ct][ks][lane]) : half8_t{};
                        const half8_t l = in ? __builtin_bit_cast(half8_t, sm.Rb[1][ct][ks][lane]) : half8_t{};
                        y = mfma16(th[ks], h, y);
                        y = mfma16(tl[ks], h, y);
                        y = mfma16(th[ks], l, y);
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) V[ct][r] = fmaf(0x1p16f, y[r], V[ct][r]);
                    put_v(ct, V[ct], dg);
                }
            }
            lds_barrier();
            // ---- 3. S = e^{G_63} S + K^T Vs ----
            if (__builtin_expect(big, 0) && lane == 0) sm.big[w] = 0;
            half8_t Vh[NC][2], Vl[NC][2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int ct = 0; ct < NC; ++ct) {
                    Vh[ct][ks] = __builtin_bit_cast(half8_t, sm.V[0][ct][ks][lane]);
                    Vl[ct][ks] = __builtin_bit_cast(half8_t, sm.V[1][ct][ks][lane]);
                }
            ahead(nx);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ct = 0; ct < NC; ++ct)
#pragma unroll
                for (int m = 0; m < 2; ++m) S[ct][m] *= ec;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int ct = 0; ct < NC; ++ct)
#pragma unroll
                    for (int m = 0; m < 2; ++m) S[ct][m] = mfma16(aK[m][ks], Vh[ct][ks], S[ct][m]);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int ct = 0; ct < NC; ++ct)
#pragma unroll
                    for (int m = 0; m < 2; ++m) {
                        S[ct][m] = mfma16(aK[m][ks], Vl[ct][ks], S[ct][m]);
                        if (kF32) S[ct][m] = mfma16(aKl[m][ks], Vh[ct][ks], S[ct][m]);
                    }
            put_state();
            lds_barrier();
        };
        put_state();
        lds_barrier();  // S written; the helpers' copy of chunk 0 is in its slot
        ahead(sm.c[0]);
        // With an odd count the helper waves take a chunk past the last one, whose operands read as
        // zero; the chain waves only meet its barriers.  (Its products would not leave the state as it
        // is: an entry above the fp16 range is infinite in the operand, and 0 * inf is NaN.)
        for (int ch = 0; ch + 1 < nch; ch += 2) {
            step(sm.c[0], sm.c[1]);
            step(sm.c[1], sm.c[0]);
        }
        if (nch & 1) {
            step(sm.c[0], sm.c[1]);
            lds_barrier();
            lds_barrier();
            lds_barrier();
        }
        bool lost = false;
        if constexpr (kFlags) {
            // a timed-out wait means some chunk operands were read before they were published:
            // beside the prep, leave the state for the second launch (sent there by the abort word,
            // cleared at the start of the call); otherwise poison it
            lds_barrier();  // the helpers' err words
            lost = (sm.err[0] | sm.err[1] | sm.err[2] | sm.err[3]) != 0;
            if (mode == kCarryBeside && tid == 0 && lost)
                __hip_atomic_store(aborts + wg, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else if (tid == 0 && unit == 0 && part < kAbortWgs) {
            // in order after the prep the abort words were not cleared: the first unit's workgroups
            // zero theirs (a workgroup that runs in order never gives up)
            __hip_atomic_store(aborts + wg, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lost && mode == kCarryBeside) return;
        const float nan = __builtin_nanf("");
#pragma unroll
        for (int ct = 0; ct < NC; ++ct)
#pragma unroll
            for (int m = 0; m < 2; ++m)
                *reinterpret_cast<float4*>((dst == state ? state + (size_t)bh * kSegSlotFloats : dst) +
                                           (size_t)col(ct, c) * kD + 32 * w + 16 * m + 4 * g) =
                    lost ? make_float4(nan, nan, nan, nan)
                         : make_float4(S[ct][m][0], S[ct][m][1], S[ct][m][2], S[ct][m][3]);
        return;
    }

    // ---- helper waves ----
    // A buffer descriptor per tensor and chunk ends with the sequence's last token (none past the
    // last chunk), so rows past the end read as zero and their stores are dropped.  Per-lane
    // offsets are fixed.
    constexpr unsigned kE = sizeof(TIO);
    const unsigned vrow = (unsigned)vs.t * kE;  // bytes between tokens of V (not with kWide)
    const TIO* vh = v + b * vs.b + (long long)c0 * kC * vs.t + h * vs.h;
    const unsigned char* wsh = ws + ((size_t)bh * nch_all + c0) * ws_chunk<kF32>();
    const unsigned char* wsq = ws + (((size_t)b * Hv + hq) * nch_all + c0) * ws_chunk<kF32>();  // the QK head's rows
    // V: 4 lanes a token, 4 NC columns a lane
    const unsigned voff = (unsigned)(16 * w + (lane >> 2)) * vrow + (unsigned)(col0 + 4 * NC * (lane & 3)) * kE;
    const unsigned lane16 = (unsigned)lane * 16;
    auto span = [&](int ch, unsigned row, unsigned last) {  // bytes of a chunk's rows
        return ch < nch ? (unsigned)(min(kC, Tloc - ch * kC) - 1) * row + last : 0u;
    };
    auto rsrc_ws = [&](const unsigned char* p, int ch) {
        return rsrc_of(p + (size_t)ch * ws_chunk<kF32>(), ch < nch ? (kF32 ? kWsUsedF32 : kWsUsed) : 0);
    };
    struct In {                 // what goes to the chain waves
        uint4 k[4], kl[kF32 ? 4 : 1], t[3];
        uint4 v[NC * (kF32 ? 2 : 1)];  // 8 bytes of it with fp16 I/O and NC = 1
        float gf;
    };
    struct Own {                // what stays: operands of this wave's tokens
        uint4 q[4], a[2];
    };
    auto load_t = [&](In& x, int ch) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t wr = rsrc_ws(wsh, ch);
#pragma unroll
        for (int j = 0; j < 3; ++j) x.t[j] = bload4w<kFlags>(wr, kWsT + (unsigned)(3 * w + j) * 1024 + lane16);
    };
    auto load_kv = [&](In& x, int ch) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t qr = rsrc_ws(wsq, ch);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x.k[j] = bload4w<kFlags>(qr, kWsK + (unsigned)(4 * w + j) * 1024 + lane16);
            if (kF32) x.kl[kF32 ? j : 0] = bload4w<kFlags>(qr, kWsKlo + (unsigned)(4 * w + j) * 1024 + lane16);
        }
        x.gf = bload1w<kFlags>(rsrc_ws(wsh, ch), kWsG + 4 * (kC * w + lane));
        if constexpr (kWide) {
            const int t = ch * kC + 16 * w + (lane >> 2);
            const uint4* p = reinterpret_cast<const uint4*>(vh + min(t, Tloc - 1) * vs.t + col0 + 4 * NC * (lane & 3));
#pragma unroll
            for (int i = 0; i < (int)(NC * kE) / 4; ++i) {
                const uint4 y = p[i];
                x.v[i] = ch < nch && t < Tloc ? y : make_uint4(0, 0, 0, 0);
            }
            return;
        }
        const __amdgpu_buffer_rsrc_t vr = rsrc_of(vh + (long long)ch * kC * vs.t, span(ch, vrow, kD * kE));
        if constexpr (NC * kE == 2) {
            const u32x2_t y = __builtin_amdgcn_raw_buffer_load_b64(vr, voff, 0, 0);
            x.v[0] = make_uint4(y[0], y[1], 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < (int)(NC * kE) / 4; ++i) x.v[i] = bload4(vr, voff + 16 * i);
        }
    };
    auto load_q = [&](Own& x, int ch) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t qr = rsrc_ws(wsq, ch);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) x.q[kk] = bload4w<kFlags>(qr, kWsQ + (unsigned)(4 * w + kk) * 1024 + lane16);
    };
    auto load_a = [&](Own& x, int ch) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t wr = rsrc_ws(wsh, ch);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) x.a[ks] = bload4w<kFlags>(wr, kWsAqk + (unsigned)(ts + min(ks, nks - 1)) * 1024 + lane16);
    };
    // (the empty asm at the end of each keeps the reloads that follow behind these uses)
    auto put_t = [&](CarrySlot<TIO, NC>& cs, const In& x) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 3; ++j) cs.T[(3 * w + j) * 64 + lane] = x.t[j];
        asm volatile("" ::: "memory");
    };
    auto put_kv = [&](CarrySlot<TIO, NC>& cs, const In& x) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int off = tile_off(16 * w + 4 * j + (lane >> 4), lane & 15);
            *reinterpret_cast<uint4*>(cs.K + off) = x.k[j];
            if (kF32) *reinterpret_cast<uint4*>(cs.K + kC * kD + off) = x.kl[kF32 ? j : 0];
        }
        TIO* vp = cs.V + (16 * w + (lane >> 2)) * 16 * NC + 4 * NC * (lane & 3);
        if constexpr (NC * kE == 2) {
            *reinterpret_cast<uint2*>(vp) = make_uint2(x.v[0].x, x.v[0].y);
        } else {
#pragma unroll
            for (int i = 0; i < (int)(NC * kE) / 4; ++i) reinterpret_cast<uint4*>(vp)[i] = x.v[i];
        }
        cs.G[kC * w + lane] = x.gf;
        asm volatile("" ::: "memory");
    };

    // Ready flags (kFlags): a wave waits for a chunk's flag before it loads the chunk's workspace.
    // After one timed-out wait, no more waits (the workgroup's results are then discarded).
    const unsigned* fl = kFlags ? flags + (size_t)bh * nch_all + c0 : nullptr;
    const unsigned* flq = kFlags ? flags + ((size_t)b * Hv + hq) * nch_all + c0 : nullptr;
    bool gave_up = false;
    auto ready = [&](int n) {
        if constexpr (kFlags) {
            auto look = [&]() {
                const unsigned f = __hip_atomic_load(fl + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const unsigned fq = __hip_atomic_load(flq + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return __builtin_amdgcn_readfirstlane(f & fq);
            };
            // real-time counter (100 MHz), low 32 bits; readfirstlane keeps the wait loop uniform
            auto now = []() { return __builtin_amdgcn_readfirstlane((unsigned)__builtin_amdgcn_s_memrealtime()); };
            if (n < nch && !gave_up && look() == 0u) {
                const unsigned t0 = now();
                while (true) {
                    if (now() - t0 >= wait_ticks) {
                        gave_up = true;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(8);
                    if (look() != 0u) break;
                }
            }
            asm volatile("" ::: "memory");  // no load of the chunk's workspace above the wait
        }
    };

    // Output rows: fp32 (fp32 I/O, or a map's rows in the workspace) or the caller's type.
    typedef typename std::conditional<kWide, size_t, unsigned>::type row_t;
    const row_t orow = obuf ? (row_t)kD * 4 : (row_t)Hv * kD * kE;
    unsigned char* ob = obuf ? reinterpret_cast<unsigned char*>(obuf)
                             : reinterpret_cast<unsigned char*>(out + (((size_t)b * T + (size_t)c0 * kC) * Hv + h) * kD);
    const bool o32 = kF32 || obuf != nullptr;  // uniform
    const unsigned ooff = (unsigned)(16 * w + c) * (unsigned)orow + (unsigned)(col0 + 4 * NC * g) * (o32 ? 4 : 2);

    // in: the next chunk's operands; o: this chunk's
    auto step = [&](In& in, Own& o, CarrySlot<TIO, NC>& cs, CarrySlot<TIO, NC>& nx, int ch) __attribute__((always_inline)) {
        // ---- 1. the next chunk's K, V and factors to the chain waves ----
        put_kv(nx, in);
        ready(ch + 3);
        load_kv(in, ch + 3);
        lds_barrier();
        // ---- 2. its T'; (Q S)^T: rows are columns of the state, so a lane ends with consecutive
        // output columns of one token ----
        half8_t Sh[NC][4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int ct = 0; ct < NC; ++ct) Sh[ct][kk] = __builtin_bit_cast(half8_t, sm.S[0][ct][kk][lane]);
        const float eq = cs.G[16 * w + c];
        put_t(nx, in);
        load_t(in, ch + 3);
        float4_t qs[NC];
#pragma unroll
        for (int ct = 0; ct < NC; ++ct) qs[ct] = float4_t{};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int ct = 0; ct < NC; ++ct)
                qs[ct] = mfma16(Sh[ct][kk], __builtin_bit_cast(half8_t, o.q[kk]), qs[ct]);
#pragma unroll
        for (int ct = 0; ct < NC; ++ct) pin(qs[ct]);
        load_q(o, ch + 2);
        lds_barrier();
        // ---- 3. O ----
        half8_t Vn[NC][2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int ct = 0; ct < NC; ++ct) Vn[ct][ks] = __builtin_bit_cast(half8_t, sm.V[2][ct][ks][lane]);
        float4_t ov[NC];
#pragma unroll
        for (int ct = 0; ct < NC; ++ct) {
            float4_t av = {};
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                if (ks >= nks) break;  // uniform
                av = mfma16(Vn[ct][ks], __builtin_bit_cast(half8_t, o.a[ks]), av);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) ov[ct][r] = scale * fmaf(eq, qs[ct][r], av[r]);
            pin(ov[ct]);
        }
        if constexpr (kWide) {
            static_assert(NC == 2, "a lane's 8 columns are one or two 16-byte stores");
            const int t = ch * kC + 16 * w + c;
            if (ch < nch && t < Tloc) {
                uint4* p = reinterpret_cast<uint4*>(ob + (size_t)t * orow + (size_t)(col0 + 4 * NC * g) * (o32 ? 4 : 2));
                if (o32) {
#pragma unroll
                    for (int ct = 0; ct < NC; ++ct) p[ct] = __builtin_bit_cast(uint4, ov[ct]);
                } else {
                    half8_t oh;
#pragma unroll
                    for (int e = 0; e < 8; ++e) oh[e] = (half_t)ov[(e >> 2) & (NC - 1)][e & 3];
                    *p = __builtin_bit_cast(uint4, oh);
                }
            }
            load_a(o, ch + 2);
            lds_barrier();
            return;
        }
        const __amdgpu_buffer_rsrc_t orr =
            rsrc_of(ob + (size_t)ch * kC * orow, span(ch, (unsigned)orow, (unsigned)kD * (o32 ? 4 : 2)));
        if (o32) {
#pragma unroll
            for (int ct = 0; ct < NC; ++ct)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, ov[ct]), orr, ooff + 16 * ct, 0, 0);
        } else {
            half4_t oh[NC];
#pragma unroll
            for (int ct = 0; ct < NC; ++ct)
#pragma unroll
                for (int r = 0; r < 4; ++r) oh[ct][r] = (half_t)ov[ct][r];
            if constexpr (NC == 2)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, cat8(oh[0], oh[NC - 1])), orr, ooff, 0, 0);
            else
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, oh[0]), orr, ooff, 0, 0);
        }
        load_a(o, ch + 2);
        lds_barrier();
    };

    In in0, in1;
    Own a0, a1;
    auto load_in = [&](In& x, int ch) __attribute__((always_inline)) {
        ready(ch);
        load_kv(x, ch);
        load_t(x, ch);
    };
    load_in(in0, 0);
    load_q(a0, 0);
    load_a(a0, 0);
    load_in(in1, 1);
    load_q(a1, 1);
    load_a(a1, 1);
    put_kv(sm.c[0], in0);
    put_t(sm.c[0], in0);
    load_in(in0, 2);
    lds_barrier();
    // chunks 0 .. 2's operands are waited for here: with loads in flight at its entry the loop's
    // own waits would be as strict as the entry's order asks for; and there is no exit between
    // the two steps, which would leave the loop's header a path with one step's loads only
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    for (int ch = 0; ch < nch; ch += 2) {
        step(in1, a0, sm.c[0], sm.c[1], ch);
        step(in0, a1, sm.c[1], sm.c[0], ch + 1);
    }
    if constexpr (kFlags) {
        if (lane == 0) sm.err[w] = gave_up;
        lds_barrier();
    }
}

// The combine of the sequence split: entry[s + 1] = Phi_s entry[s] + Z_s for s = 1 .. nseg - 1,
// in fp32; entry[nseg] is the call's final state (state, same layout).  Slots are stored [column][dk]; row j of the Phi slot is Phi's column j, so with
// E = entry[s] stored the same way, entry[s + 1][c][d] = sum_j E[c][j] Phi[j][d] + Z[c][d].
// State columns never mix: a workgroup takes R columns of one head through every step and
// waits for no other workgroup.  Only the E chain is serial: wave w sums over j in
// [32 w, 32 w + 32) with its lane's dk pair (2 lane, 2 lane + 1), holding that quarter of
// Phi_s in registers while the next step's quarter loads; the four partial sums meet in LDS.
// Every workgroup reads all of Phi_s per step whatever R is, while its FMA time grows with R:
// the host picks the smallest R that keeps about one workgroup per CU.
constexpr int kCombThreads = 256;
template <int R>
__global__ void __launch_bounds__(kCombThreads) gdn_seg_combine(float* __restrict__ seg, float* __restrict__ state,
                                                                int nseg) {
    const int bh = blockIdx.x / (kD / R), c0 = (blockIdx.x % (kD / R)) * R;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    float* segh = seg + (size_t)bh * nseg * kSegSlots * kSegSlotFloats;
    auto slot = [&](int sg, int which) { return segh + ((size_t)sg * kSegSlots + which) * kSegSlotFloats; };
    constexpr int kOut = (R * kD + kCombThreads - 1) / kCombThreads;  // outputs per thread
    __shared__ __align__(16) float E[R][kD];
    __shared__ __align__(16) float part[4][R][kD];
    if (tid < R * kD / 4)
        reinterpret_cast<float4*>(&E[0][0])[tid] =
            reinterpret_cast<const float4*>(slot(1, kSegEntry) + (size_t)c0 * kD)[tid];
    auto quarter = [&](int sg, float2 (&p)[32]) {
        const float2* P = reinterpret_cast<const float2*>(slot(sg, kSegPhi) + (size_t)(32 * w) * kD) + lane;
#pragma unroll
        for (int jj = 0; jj < 32; ++jj) p[jj] = P[jj * (kD / 2)];
    };
    // this thread's outputs in the reduction: o = tid + 256 i < R * 128 is (row o / 128, dk o % 128)
    auto zload = [&](int sg, float (&z)[kOut]) {
        const float* Z = slot(sg, kSegZ) + (size_t)c0 * kD;
#pragma unroll
        for (int i = 0; i < kOut; ++i) z[i] = Z[min(tid + kCombThreads * i, R * kD - 1)];
    };
    // step sg computes with (pc, zc) while step sg + 1's quarter loads into (pn, zn); the loop
    // is unrolled by two so the two register sets swap roles without copies
    auto step = [&](int sg, const float2 (&pc)[32], const float (&zc)[kOut], float2 (&pn)[32], float (&zn)[kOut]) {
        // unconditional (the last step reloads its own slot): a branch around the loads would
        // make the compiler wait for them where the paths join
        const int nx = min(sg + 1, nseg - 1);
        quarter(nx, pn);
        zload(nx, zn);
        float2 acc[R] = {};
#pragma unroll
        for (int jj = 0; jj < 32; jj += 4) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float4 e = *reinterpret_cast<const float4*>(&E[r][32 * w + jj]);
                acc[r].x = fmaf(e.x, pc[jj].x, acc[r].x);
                acc[r].y = fmaf(e.x, pc[jj].y, acc[r].y);
                acc[r].x = fmaf(e.y, pc[jj + 1].x, acc[r].x);
                acc[r].y = fmaf(e.y, pc[jj + 1].y, acc[r].y);
                acc[r].x = fmaf(e.z, pc[jj + 2].x, acc[r].x);
                acc[r].y = fmaf(e.z, pc[jj + 2].y, acc[r].y);
                acc[r].x = fmaf(e.w, pc[jj + 3].x, acc[r].x);
                acc[r].y = fmaf(e.w, pc[jj + 3].y, acc[r].y);
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) *reinterpret_cast<float2*>(&part[w][r][2 * lane]) = acc[r];
        __syncthreads();  // partial sums written, E read by every wave
        float* en = (sg + 1 < nseg ? slot(sg + 1, kSegEntry) : state + (size_t)bh * kSegSlotFloats) + (size_t)c0 * kD;
#pragma unroll
        for (int i = 0; i < kOut; ++i) {
            const int o = tid + kCombThreads * i, r = o / kD, d = o % kD;
            if (o < R * kD) {
                const float v = zc[i] + part[0][r][d] + part[1][r][d] + part[2][r][d] + part[3][r][d];
                E[r][d] = v;
                en[o] = v;
            }
        }
        __syncthreads();
    };
    float2 pa[32], pb[32];
    float za[kOut], zb[kOut];
    quarter(1, pa);
    zload(1, za);
    __syncthreads();
    for (int sg = 1; sg < nseg; sg += 2) {
        step(sg, pa, za, pb, zb);
        if (sg + 1 >= nseg) break;
        step(sg + 1, pb, zb, pa, za);
    }
}

// The fixup of the sequence split: O = O_Z + M E^T for the tokens of segments 1 .. nseg-1,
// every chunk in parallel (a workgroup per (b, h, chunk)).  M [token][dk] and O_Z
// [token][column] are the map chains' fp32 outputs (scale included), E [column][dk] the
// entry state of the chunk's segment.  The product runs on fp16 MFMAs with each fp32 operand
// as an exact hi + lo pair (hi hi + hi lo + lo hi).  E goes to LDS as the B operands' hi and lo
// halves, rows padded to kFixRow halfs so that the 16 rows one read touches fall in different
// banks; wave w takes tokens 16 (w % 4) .. + 15 of the chunk and columns 64 (w / 4) .. + 63.
constexpr int kFixRow = kD + 8;
constexpr int kFixThreads = 512;
template <typename TIO>
__global__ void __launch_bounds__(kFixThreads)
gdn_seg_fixup(const float* __restrict__ seg, const float* __restrict__ oz, const float* __restrict__ om,
              TIO* __restrict__ out, int T, int Hv, int nseg, int seg_len, int Tr, int nfix) {
    const int bh = blockIdx.x / nfix, cl = blockIdx.x % nfix;  // cl: chunk counted from segment 1's start
    const int b = bh / Hv, h = bh % Hv;
    const int sg = min(seg_len + cl, nseg * seg_len - 1) / seg_len;  // the chunk's segment (1 .. nseg-1)
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int w = (tid >> 6) & 3, n0 = 4 * (tid >> 8);  // token block; first 16-column tile
    __shared__ __align__(16) half_t Eh[kD * kFixRow];
    __shared__ __align__(16) half_t El[kD * kFixRow];
    // Every global load is issued before any is used (E's 16 float4s per thread, this lane's
    // M row, its 16 O_Z values), from clamped addresses, and only the stores are guarded: a
    // load behind a branch, or one per loop trip between LDS stores, waits out its own memory
    // latency.
    const float* E = seg + ((size_t)bh * nseg * kSegSlots + (size_t)sg * kSegSlots + kSegEntry) * kSegSlotFloats;
    constexpr int kEPer = kD * kD / 4 / kFixThreads;  // float4s of E per thread
    float4 ev[kEPer];
#pragma unroll
    for (int i = 0; i < kEPer; ++i) ev[i] = reinterpret_cast<const float4*>(E)[tid + kFixThreads * i];
    // A operands: this lane's token row of M (rows past T, which the buffers do not hold, read
    // the last row and are not stored), dk 32 ks + 8 g .. + 7
    const size_t base = (size_t)bh * Tr;
    const size_t ra = base + min((size_t)cl * kC + 16 * w + c, (size_t)Tr - 1);
    float4 mv[4][2];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const float4* mp = reinterpret_cast<const float4*>(om + ra * kD + 32 * ks + 8 * g);
        mv[ks][0] = mp[0];
        mv[ks][1] = mp[1];
    }
    // O_Z of this lane's outputs: tokens 16 w + 4 g + r, columns 16 (n0 + nt) + c
    float zv[4][4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            zv[nt][r] = oz[(base + min((size_t)cl * kC + 16 * w + 4 * g + r, (size_t)Tr - 1)) * kD + 16 * (n0 + nt) + c];
#pragma unroll
    for (int i = 0; i < kEPer; ++i) {
        const float e4[4] = {ev[i].x, ev[i].y, ev[i].z, ev[i].w};
        half4_t hv, lv;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            hv[q] = (half_t)e4[q];
            lv[q] = (half_t)(e4[q] - (float)hv[q]);
        }
        const int f = 4 * (tid + kFixThreads * i), row = f / kD, col = f % kD;
        *reinterpret_cast<half4_t*>(&Eh[row * kFixRow + col]) = hv;
        *reinterpret_cast<half4_t*>(&El[row * kFixRow + col]) = lv;
    }
    half8_t ah[4], al[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const float m8[8] = {mv[ks][0].x, mv[ks][0].y, mv[ks][0].z, mv[ks][0].w,
                             mv[ks][1].x, mv[ks][1].y, mv[ks][1].z, mv[ks][1].w};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            ah[ks][q] = (half_t)m8[q];
            al[ks][q] = (half_t)(m8[q] - (float)ah[ks][q]);
        }
    }
    __syncthreads();
    const int t0 = (seg_len + cl) * kC;  // the chunk's first token
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        float4_t acc = {};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int o = (16 * (n0 + nt) + c) * kFixRow + 32 * ks + 8 * g;
            const half8_t bhv = *reinterpret_cast<const half8_t*>(&Eh[o]);
            const half8_t blv = *reinterpret_cast<const half8_t*>(&El[o]);
            acc = mfma16(ah[ks], bhv, acc);
            acc = mfma16(ah[ks], blv, acc);
            acc = mfma16(al[ks], bhv, acc);
        }
        // acc[r]: token 16 w + 4 g + r, column 16 (n0 + nt) + c
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int tl = 16 * w + 4 * g + r;
            if (t0 + tl < T)
                out[(((size_t)b * T + t0 + tl) * Hv + h) * kD + 16 * (n0 + nt) + c] = (TIO)(zv[nt][r] + acc[r]);
        }
    }
}

// Clears the ready flags and abort words of a call (n words) before anything reads them.
__global__ void __launch_bounds__(256) gdn_flags_clear(unsigned* __restrict__ w, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) w[i] = 0u;
}

// A positive integer from the environment, or `def` when unset or malformed.
long env_long(const char* name, long def, long hi) {
    const char* e = std::getenv(name);
    if (!e || !*e) return def;
    char* end = nullptr;
    const long v = std::strtol(e, &end, 10);
    return (end && *end == 0 && v >= 0 && v <= hi) ? v : def;
}

// The sequence split of a call: nseg segments of seg_len chunks (nseg == 1: no split).  It pays
// where the carry's workgroups leave most CUs idle (few heads) and the chunk chain is long.
// The call's serial time is about nch / nseg chunk steps (the maps) + nseg - 1 combine steps
// (each about a chunk step) + the fixup, least near nseg = sqrt(nch); the library's plan
// (req = 0) takes the most segments up to sqrt(nch) whose maps launch ((2 nseg - 1) units of 4
// workgroups per head) fits in the 256 CUs of the part, each at least kMinSegChunks chunks
// long: a function of the shapes only, so a workspace sized once serves every call of a shape.
// An explicit request (tsa_gdn_chunked_plan_fwd) replaces it: req = 1 never splits, req >= 2
// asks for req segments (fewer if the sequence has fewer chunks: no segment is empty).
// us per call, fp16, no split / this plan / the best of 1 to 8 segments: T = 4096 1 head 63.4 / 35.8 / 35.8,
// 4 heads 63.6 / 44.3 / 40.9 (4 segments), 8 67.1 / 55.4 / 54.8, 16 70.2 / 78.0 / 70.2; T = 2048 1 head 38.0 /
// 30.9, 4 37.8 / 34.5, 8 38.3 / 40.6, 16 39.9 / 49.1; T = 1536 4 31.1 / 32.2; T = 1024 1 24.9 / 28.1, 4 24.6 / 29.5, 16
// 25.5 / 39.7; T = 16384 4 229 / 97.  The plan was set for carry steps of 32 columns alone; an unsplit
// carry of few heads now takes 16, so up to 16 chunks, and from 8 to 16 heads on, the plan is
// the slower one (with the carry it was set for, T = 1024, 4 heads took 52 unsplit and 35.6 split).
constexpr int kSplitCUs = 256;
constexpr int kMinSegChunks = 8;
struct SegPlan {
    int nseg = 1, seg_len = 0;
};
SegPlan seg_plan(int BHv, int nch, int req) {
    long n = 1;
    if (req >= 2)
        n = std::min<long>(req, nch);
    else if (req == 0 && BHv > 0)
        n = std::min<long>(std::min<long>((kSplitCUs / (4 * BHv) + 1) / 2, nch / kMinSegChunks),
                           (long)std::sqrt((double)nch));
    if (n < 2) return {};
    const int seg_len = (int)((nch + n - 1) / n);
    n = (nch + seg_len - 1) / seg_len;  // no empty segment
    if (n < 2) return {};
    return {(int)n, seg_len};
}

// Byte offset of the split's slots in the workspace: after the chunk workspaces, the ready
// flags and the abort words, rounded up to 256 B.
size_t seg_offset(size_t BHv, size_t nch, bool f32) {
    const size_t end = BHv * nch * ((f32 ? kWsChunkF32 : kWsChunk) + sizeof(unsigned)) +
                       BHv * kAbortWgs * sizeof(unsigned);
    return (end + 255) & ~(size_t)255;
}
}  // namespace

namespace {
// Workspace bytes of a call under a plan: chunk workspaces, then a ready flag per chunk, then
// an abort word per carry workgroup, then, when the call splits, the slots and the maps' O_Z
// and M rows of the tokens after segment 0
size_t ws_bytes_for(size_t BHv, size_t nch, int T, bool f32, const SegPlan& plan) {
    if (plan.nseg == 1)
        return BHv * nch * ((f32 ? kWsChunkF32 : kWsChunk) + sizeof(unsigned)) +
               BHv * kAbortWgs * sizeof(unsigned);
    const size_t Tr = (size_t)T - (size_t)plan.seg_len * kC;
    return seg_offset(BHv, nch, f32) + BHv * plan.nseg * kSegSlots * kSegSlotFloats * sizeof(float) +
           2 * BHv * Tr * kD * sizeof(float);
}

// The plan of a call whose workspace holds at most `budget` bytes: the split where it fits,
// else none (the no-allocation entry's fixed scratch).
SegPlan call_plan(int BHv, int nch, int T, bool f32, size_t budget, int req) {
    SegPlan plan = seg_plan(BHv, nch, req);
    if (plan.nseg > 1 && ws_bytes_for((size_t)BHv, (size_t)nch, T, f32, plan) > budget) plan = SegPlan{};
    return plan;
}
}  // namespace

size_t gdn_chunked_ws_bytes(int B, int T, int Hv, bool f32, int nseg) {
    const int nch = (T + kC - 1) / kC, BHv = B * Hv;
    return ws_bytes_for((size_t)BHv, (size_t)nch, T, f32, call_plan(BHv, nch, T, f32, SIZE_MAX, nseg));
}

namespace {

// With TSA_GDN_OVERLAP=1 the prep runs on a second stream of the device so that it overlaps
// the carry: the carry copies a chunk's operands as soon as the prep has published them
// (ready flags), and the chunk-major prep order produces them in the order the carry consumes
// them.  One side stream and its fork / join events per device, created on the first call
// that overlaps on that device and kept until the process ends.
struct SideStream {
    bool tried = false, ok = false;
    int cus = 0;
    hipStream_t s = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
};
constexpr int kMaxDevices = 64;
std::mutex g_side_mu;
SideStream g_side[kMaxDevices];

// Longest wait of a carry workgroup for a chunk, in ticks of the 100 MHz real-time counter.
unsigned carry_wait_ticks() { return (unsigned)(env_long("TSA_GDN_CARRY_WAIT_US", 2000, 10000000) * 100); }

// The prep and the carry run in order on the caller's stream unless the environment variable
// TSA_GDN_OVERLAP=1 asks for the side-by-side form (the prep on a second stream, the carry
// waiting on its ready flags).  In order is the default: at 32 heads it measured as fast as
// the overlap, and it needs no side stream, events, mutex, flag clear or second carry launch.
bool overlap_requested() { return env_long("TSA_GDN_OVERLAP", 0, 1) != 0; }

template <bool kFused, typename TIO>
hipError_t launch_chunked(const void* q, const void* k, const void* v, const float* g_log,
                          const float* beta, const GdnRawGates& gates, const float* state_in, float* state,
                          void* out, int B, int T, int Hq, int Hv, float scale, void* ws, bool may_overlap,
                          hipStream_t stream, const GdnStrides& st, size_t ws_budget = SIZE_MAX, int nseg = 0) {
    const int nch = (T + kC - 1) / kC;
    const int BHv = B * Hv;
    const int carry_wgs = BHv * kAbortWgs;
    auto Q = static_cast<const TIO*>(q);
    auto K = static_cast<const TIO*>(k);
    auto V = static_cast<const TIO*>(v);
    auto W = static_cast<unsigned char*>(ws);
    unsigned* flags = reinterpret_cast<unsigned*>(W + (size_t)BHv * nch * ws_chunk<std::is_same<TIO, float>::value>());
    unsigned* aborts = flags + (size_t)BHv * nch;
    const int nflags = BHv * nch + carry_wgs;
    const unsigned wait_ticks = carry_wait_ticks();
    // a chunk's 64 rows of V or the output are out of a buffer descriptor's reach
    const bool wide = std::max(st.v.t, (long long)Hv * kD) > INT_MAX / kC / (long long)sizeof(TIO);
    auto clear = [&]() {
        hipLaunchKernelGGL(gdn_flags_clear, dim3((nflags + 255) / 256), dim3(256), 0, stream, flags, nflags);
        return hipGetLastError();
    };
    // In order (the prep, then the carry, on one stream) no ready flags are written or read.
    auto prep = [&](hipStream_t on, bool publish) {
        hipLaunchKernelGGL((gdn_chunk_prep<kFused, TIO>), dim3(BHv * nch), dim3(kThreads), 0, on, Q, K,
                           g_log, beta, gates, W, publish ? flags : nullptr, T,
                           Hq, Hv, nch, BHv, st);
        return hipGetLastError();
    };
    auto carry = [&](int mode, unsigned ticks, int units = 1, CarryJob job = CarryJob{}) {
        auto launch = [&](auto kernel, int wgs) {
            hipLaunchKernelGGL(kernel, dim3(units == 1 ? wgs * ((BHv + 7) & ~7) : units * wgs * BHv), dim3(kCarryThreads), 0, stream, V, W,
                               mode == kCarryInOrder ? nullptr : flags, aborts, mode, ticks, state_in,
                               state, static_cast<TIO*>(out), T, Hq, Hv, nch, BHv, scale, job, st.v);
            return hipGetLastError();
        };
        if (mode != kCarryInOrder) return launch(gdn_chunk_carry<TIO, 2, true>, kAbortWgs);
        if (wide) return launch(gdn_chunk_carry<TIO, 2, false, true>, kAbortWgs);
        // A workgroup takes a CU.  16 columns each while every workgroup then has a CU of its own,
        // else 32: a chunk step of 32 columns is ~1.25 steps of 16, and a second round costs a
        // whole one.  (us per carry, 16 / 32 columns: 32 heads, T = 4096 74 / 88; 48 heads, T = 1000
        // 36 / 27; fp32 I/O, 48 heads, T = 512 30 / 22; maps of 4 heads, T = 4096 23 / 18.)
        if (units * 2 * kAbortWgs * BHv <= kSplitCUs) return launch(gdn_chunk_carry<TIO, 1, false>, 2 * kAbortWgs);
        return launch(gdn_chunk_carry<TIO, 2, false>, kAbortWgs);
    };

    // Sequence split: in order on the caller's stream (the maps need every chunk's operands)
    const SegPlan plan = call_plan(BHv, nch, T, std::is_same<TIO, float>::value, ws_budget, nseg);
    if (plan.nseg > 1) {
        CarryJob job;
        job.phase = kJobMaps;
        job.nseg = plan.nseg;
        job.seg_len = plan.seg_len;
        job.Tr = T - plan.seg_len * kC;
        job.seg = reinterpret_cast<float*>(W + seg_offset(BHv, nch, std::is_same<TIO, float>::value));
        job.oz = job.seg + (size_t)BHv * plan.nseg * kSegSlots * kSegSlotFloats;
        job.om = job.oz + (size_t)BHv * job.Tr * kD;
        hipError_t e = prep(stream, false);
        if (e == hipSuccess) e = carry(kCarryInOrder, wait_ticks, 2 * plan.nseg - 1, job);
        if (e == hipSuccess) {
            // state columns per combine workgroup: about one workgroup per CU
            const int rows = BHv <= 2 ? 1 : BHv <= 4 ? 2 : BHv <= 8 ? 4 : 8;
            auto combine = rows == 1 ? gdn_seg_combine<1> : rows == 2 ? gdn_seg_combine<2>
                         : rows == 4 ? gdn_seg_combine<4> : gdn_seg_combine<8>;
            hipLaunchKernelGGL(combine, dim3(BHv * (kD / rows)), dim3(kCombThreads), 0, stream, job.seg, state,
                               plan.nseg);
            e = hipGetLastError();
        }
        if (e == hipSuccess) {
            const int nfix = nch - plan.seg_len;
            hipLaunchKernelGGL(gdn_seg_fixup<TIO>, dim3(BHv * nfix), dim3(kFixThreads), 0, stream, job.seg, job.oz,
                               job.om, static_cast<TIO*>(out), T, Hv, plan.nseg, plan.seg_len, job.Tr, nfix);
            e = hipGetLastError();
        }
        return e;
    }

    // The default, and every call that cannot overlap: in order on the caller's stream, with no
    // other runtime call.  The overlap (TSA_GDN_OVERLAP=1) is taken only when it cannot stall:
    // the carry's workgroups (one per CU) must leave at least half the CUs to the prep, and a
    // stream being captured into a graph runs the two kernels in order (a graph does not promise
    // to run sibling nodes concurrently), and so does an output that lies on v: a workgroup that
    // gives up beside the prep has written output rows, and the second launch reads V again.  The side stream belongs to the device of the caller's
    // stream (the null stream: the current device), which need not be the current device.
    hipStreamCaptureStatus cap = hipStreamCaptureStatusActive;
    int dev = -1;
    SideStream* side = nullptr;
    auto v_end = V + (B - 1) * st.v.b + (T - 1) * st.v.t + (Hv - 1) * st.v.h + kD;
    auto O = static_cast<const TIO*>(out);
    const bool on_v = O < v_end && V < O + (size_t)B * T * Hv * kD;
    if (may_overlap && !wide && !on_v && nch > 1 && overlap_requested() && hipStreamIsCapturing(stream, &cap) == hipSuccess &&
        cap == hipStreamCaptureStatusNone &&
        (stream ? hipStreamGetDevice(stream, &dev) == hipSuccess : hipGetDevice(&dev) == hipSuccess) &&
        dev >= 0 && dev < kMaxDevices) {
        std::lock_guard<std::mutex> lock(g_side_mu);
        SideStream& d = g_side[dev];
        if (!d.tried) {  // create the stream and events on that device
            d.tried = true;
            int cur = -1;
            const bool switched = hipGetDevice(&cur) == hipSuccess && cur != dev && hipSetDevice(dev) == hipSuccess;
            d.ok = (cur == dev || switched) &&
                   hipDeviceGetAttribute(&d.cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
                   hipStreamCreateWithFlags(&d.s, hipStreamNonBlocking) == hipSuccess &&
                   hipEventCreateWithFlags(&d.fork, hipEventDisableTiming) == hipSuccess &&
                   hipEventCreateWithFlags(&d.join, hipEventDisableTiming) == hipSuccess;
            if (switched) (void)hipSetDevice(cur);
        }
        if (d.ok && 2 * carry_wgs <= d.cus) side = &d;
    }
    if (!side) {  // in order: no flag clear needed
        const hipError_t e = prep(stream, false);
        return e != hipSuccess ? e : carry(kCarryInOrder, wait_ticks);
    }
    hipError_t e = clear();
    if (e != hipSuccess) return e;
    // fork: the prep starts after the caller's earlier work (the flag clear included); the
    // carry is queued first so its workgroups take their CUs before the prep fills the rest.
    // join: the caller's stream waits for the prep, then the second carry launch redoes any
    // workgroup that gave up (and otherwise exits at once).  The second launch must stay
    // behind the join: under a scheduler that serialises dispatches it could otherwise run
    // before the prep and wait for flags that cannot come.
    std::lock_guard<std::mutex> lock(g_side_mu);
    e = hipEventRecord(side->fork, stream);
    if (e == hipSuccess) e = hipStreamWaitEvent(side->s, side->fork, 0);
    if (e == hipSuccess) e = carry(kCarryBeside, wait_ticks);
    if (e == hipSuccess) e = prep(side->s, true);
    if (e == hipSuccess) e = hipEventRecord(side->join, side->s);
    if (e == hipSuccess) e = hipStreamWaitEvent(stream, side->join, 0);
    if (e == hipSuccess) e = carry(kCarryRetry, kRetryWaitTicks);
    return e;
}
}  // namespace

// ---- the no-allocation variant ----
// `scratch` stands in for the caller's workspace: a file-scope device array that each GPU the
// library runs on holds from the module's load until the process ends.  Host code never
// passes the array's name to a kernel (on the host it is only a stand-in for the symbol):
// the device address comes from hipGetSymbolAddress, once per device, on the first call on
// that device, and is kept in g_scratch.  Every call on a GPU shares that GPU's array and
// leaves its contents behind: the call runs the prep and the carry in order, so it reads no
// ready flags, the carry zeroes the abort words, and the rest of the workspace is written
// before it is read.  Calls that overlap on one GPU race on the
// array.
constexpr size_t kScratchBytes = 64ull << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
std::mutex g_scratch_mu;
void* g_scratch[kMaxDevices];

hipError_t scratch_address(hipStream_t stream, void** out) {
    int dev = -1;
    hipError_t e = stream ? hipStreamGetDevice(stream, &dev) : hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {  // with that device current
        int cur = -1;
        if ((e = hipGetDevice(&cur)) != hipSuccess) return e;
        if (cur != dev && (e = hipSetDevice(dev)) != hipSuccess) return e;
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != dev) (void)hipSetDevice(cur);
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch[dev] = p;
    }
    *out = g_scratch[dev];
    return hipSuccess;
}
}  // namespace

size_t gdn_chunked_noalloc_max_bytes() { return kScratchBytes; }

// The no-allocation entry splits the sequence only where the split's workspace fits the scratch.
size_t gdn_chunked_noalloc_ws_bytes(int B, int T, int Hv) {
    const int nch = (T + kC - 1) / kC, BHv = B * Hv;
    return ws_bytes_for((size_t)BHv, (size_t)nch, T, false, call_plan(BHv, nch, T, false, kScratchBytes, 0));
}

hipError_t gdn_chunked_noalloc(const void* q, const void* k, const void* v, const float* g_log,
                               const float* beta, float* state, void* out, int B, int T, int Hq,
                               int Hv, float scale, hipStream_t stream) {
    void* ws = nullptr;
    const hipError_t e = scratch_address(stream, &ws);
    if (e != hipSuccess) return e;
    // in order on the caller's stream: no side stream or event is ever created here
    return launch_chunked<false, half_t>(q, k, v, g_log, beta, GdnRawGates{}, state, state, out, B, T, Hq, Hv,
                                         scale, ws, false, stream, gdn_dense(T, Hq, Hv), kScratchBytes);
}

hipError_t gdn_chunked_redo_count(const void* ws, int B, int T, int Hv, bool f32, int* count,
                                  hipStream_t stream) {
    const size_t nch = (size_t)(T + kC - 1) / kC;
    const size_t n = (size_t)B * Hv * kAbortWgs;
    const unsigned char* aborts = static_cast<const unsigned char*>(ws) +
                                  (size_t)B * Hv * nch * ((f32 ? kWsChunkF32 : kWsChunk) + sizeof(unsigned));
    unsigned* host = static_cast<unsigned*>(std::malloc(n * sizeof(unsigned)));
    if (!host) return hipErrorOutOfMemory;
    hipError_t e = hipMemcpyAsync(host, aborts, n * sizeof(unsigned), hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e == hipSuccess) {
        int c = 0;
        for (size_t i = 0; i < n; ++i) c += host[i] != 0u;
        *count = c;
    }
    std::free(host);
    return e;
}

hipError_t gdn_chunked(const void* q, const void* k, const void* v, const float* g_log,
                       const float* beta, float* state, void* out, int B, int T, int Hq, int Hv,
                       float scale, void* ws, bool f32, hipStream_t stream, int nseg) {
    const GdnStrides st = gdn_dense(T, Hq, Hv);
    if (f32)
        return launch_chunked<false, float>(q, k, v, g_log, beta, GdnRawGates{}, state, state, out, B, T, Hq,
                                            Hv, scale, ws, true, stream, st, SIZE_MAX, nseg);
    return launch_chunked<false, half_t>(q, k, v, g_log, beta, GdnRawGates{}, state, state, out, B, T, Hq,
                                         Hv, scale, ws, true, stream, st, SIZE_MAX, nseg);
}

hipError_t gdn_chunked_strided(const void* q, const void* k, const void* v, const GdnStrides& st,
                               const float* g_log, const float* beta, const float* state_in, float* state,
                               void* out, int B, int T, int Hq, int Hv, float scale, void* ws, bool f32,
                               hipStream_t stream) {
    if (f32)
        return launch_chunked<false, float>(q, k, v, g_log, beta, GdnRawGates{}, state_in, state, out, B, T, Hq,
                                            Hv, scale, ws, true, stream, st);
    return launch_chunked<false, half_t>(q, k, v, g_log, beta, GdnRawGates{}, state_in, state, out, B, T, Hq,
                                         Hv, scale, ws, true, stream, st);
}

hipError_t gdn_chunked_fused(const void* q, const void* k, const void* v, const GdnRawGates& gates,
                             float* state, void* out, int B, int T, int Hq, int Hv, float scale,
                             void* ws, hipStream_t stream) {
    return launch_chunked<true, half_t>(q, k, v, nullptr, nullptr, gates, state, state, out, B, T, Hq, Hv,
                                        scale, ws, true, stream, gdn_dense(T, Hq, Hv));
}

}  // namespace tsa
