// Batch-1 greedy TDT decode in one persistent launch: 2-layer LSTM prediction
// network (gate rows i, f, g, o of 4H), projection + bias, joint, token /
// duration decision and the frame / symbol rules, for all frames of one
// utterance.  Two prediction-network forms, as in the reference:
//  - fp16 (decoder.cu:146-445, tdt_persistent_fp16): fp16 weights, fp32 state;
//  - long (decoder.cu:452-784, tdt_persistent_fp8, used for utterances of
//    1024 frames and more, decoder.rs:15,86-92): W_hh of both layers and W_ih
//    of layer 1 as per-tensor symmetric INT8 derived inside the launch
//    (scale = max|w| / 127), hidden states carried as INT8 at a fixed 1/127
//    scale next to the fp32 ones, layer 0's input terms read from a
//    [tokens x 4H] fp16 table (embedding x W_ih0^T), and the recurrent terms of
//    the state the next update consumes summed as soon as that state exists.
//
// Every weight stays in registers for the whole decode: the grid is one
// workgroup per CU (up to 256, 4 wave64 each) and wave w owns LSTM hidden unit
// w of both layers (4 gates x (W_ih, W_hh) rows), projection row w and joint
// rows 2w, 2w+1 (logical order: the duration rows first, so workgroup 0 holds
// them all).  Lane l holds k = 2l + 128j (j < H/128) of every row it owns.
// The phases (layer 0, layer 1, projection, joint) are separated by a grid
// barrier made of per-workgroup published 64-bit words (a step tag and, for
// the joint, the workgroup's best token key and workgroup 0's duration): every
// workgroup polls all words in parallel, so one barrier costs about one memory
// round trip, and the joint's decision comes with its barrier.  State vectors
// (h, c of both layers, double buffered as committed / candidate, and the
// prediction) move through agent-scope atomic stores and loads in a caller
// workspace.  Blank steps run only the joint; an emitted token commits the
// candidate state and re-runs the prediction network on its embedding.
//
// Long form: lane l holds bytes 4l + 256j (j < ceil(H/256)) of every INT8
// row; a gate's INT8 dot product is summed exactly as an integer over the
// wave (|sum| <= H * 127 * 127 < 2^24), converted once and scaled by
// scale / 127.  Layer 0 needs no weights of its own once its recurrent sums
// are known (its input terms are table rows), so every workgroup evaluates all
// of its units as soon as the token is decided and goes straight on to layer
// 1: an update costs two grid barriers (after layer 1, after the projection),
// not three.  The recurrent sums of a candidate state are taken as soon as
// that state exists (layer 0's next to layer 1, layer 1's in the projection
// phase) and used by the update after a token commits it.  Layer 1's cell
// state stays in the owning wave's registers, layer 0's in every thread that
// evaluates the unit; the INT8 layer-1 banks, the candidate fp32 layer-1
// output, the layer-0 sums and the prediction go through the workspace.
#include "pk_cell.hpp"
#include "pk_decision.hpp"
#include "pk_kernels.hpp"

namespace pk {

namespace {

constexpr int kDecThreads = 256;
constexpr int kDecMaxBlocks = 256;
constexpr uint32_t kDecSpinLimit = 1u << 22;
constexpr int kDecWords = 8;                                // u32 offset of the barrier words
constexpr int kDecState = kDecWords + 2 * kDecMaxBlocks * 2;  // u32 offset of the state vectors, after the words
static_assert(kDecState == 1032, "workspace layout");
// Frames a joint round scores against one prediction (its window), and the
// words of the joint rounds' barrier: per workgroup one key per window frame,
// each carrying the barrier tag (2 epoch slots x kWin x 256 u64, word-major so
// that the poll reads consecutive words), after the state vectors.
constexpr int kWin = 8;
constexpr int kDecExtWords = 2 * kDecMaxBlocks * kWin * 2;

struct DecodeArgs {
    const uint16_t* enc;    // [frames x enc_stride] fp16
    const uint16_t* emb;    // [token_outputs - 1 x H] fp16 (fp16 form)
    const uint16_t* table;  // [token_outputs - 1 x 4H] fp16 layer-0 input terms (long form)
    const uint16_t* w_ih[2];
    const uint16_t* w_hh[2];
    const float* b_ih[2];
    const float* b_hh[2];
    const uint16_t* w_proj;
    const float* b_proj;
    const void* w_joint;  // fp16 or int8 [outputs x H]
    const float* joint_scales;
    const float* b_joint;
    int32_t* tokens;
    int32_t* result;  // {tokens emitted, final frame, status, joint steps}
    uint32_t* ws;     // [0] abort; words at kDecWords (2 x 256 u64 = 1024 u32); state floats at kDecState
    int frames, enc_stride, outputs, token_outputs, durations, max_symbols, capacity;
};

__device__ __forceinline__ uint32_t key_bits(float score) {
    if (score == 0.0f) score = 0.0f;
    const uint32_t bits = __float_as_uint(score);
    return (bits & 0x80000000u) ? ~bits : (bits ^ 0x80000000u);
}

__device__ __forceinline__ float sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }

__device__ __forceinline__ float2 ld2(const float* p) {
    const unsigned long long v = __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
}
__device__ __forceinline__ float ld1(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void st1(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v = add_level(v, off);
    return v;
}
__device__ __forceinline__ int wave_isum(int v) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v = add_level(v, off);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v = max_level(v, off);
    return v;
}

// decoder.cu:95-97 quantize_i8: round to nearest even, clamp to +-127.
__device__ __forceinline__ int quant_i8(float v) { return max(-127, min(127, (int)__builtin_rintf(v))); }

__device__ __forceinline__ uint32_t ld_word(const uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void st_word(uint32_t* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// fp16 pair -> two floats
__device__ __forceinline__ float lo16(uint32_t w) { return h2f((uint16_t)(w & 0xffffu)); }
__device__ __forceinline__ float hi16(uint32_t w) { return h2f((uint16_t)(w >> 16)); }

template <bool kInt8, int KP, bool kLong>
__global__ __launch_bounds__(kDecThreads, 1) void tdt_decode_kernel(DecodeArgs p) {
    constexpr int H = 128 * KP;
    constexpr int KD = (KP + 1) / 2;  // INT8 dwords per lane and row (long form)
    __shared__ float red_s[12];
    __shared__ uint32_t qb_s[4];
    __shared__ float dur_sc[kWin][8];
    __shared__ unsigned long long win_w[4][kWin];  // per wave, then the decided key per window frame
    __shared__ int win_tok[kWin], win_dur[kWin];
    __shared__ int stop_s;
    // long form: the new INT8 layer-0 output, computed whole by every workgroup
    __shared__ uint32_t q0_s[kLong ? H / 4 : 1];
    const int blk = blockIdx.x, nblocks = gridDim.x;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int gw = blk * 4 + wave;
    const int T = p.token_outputs, D = p.durations, blank = T - 1;
    unsigned long long* words = (unsigned long long*)(p.ws + kDecWords);
    float* st = (float*)(p.ws + kDecState);
    // state: h[buf][layer][H], c[buf][layer][H], pred[H]
    auto hp = [&](int buf, int layer) { return st + (buf * 2 + layer) * H; };
    auto cp = [&](int buf, int layer) { return st + 4 * H + (buf * 2 + layer) * H; };
    float* pred = st + 8 * H;
    // long form: INT8 hidden vectors [bank][layer][H] bytes, candidate fp32
    // layer-1 output, per-workgroup weight maxima [blocks][3]
    uint32_t* qh = p.ws + kDecState;
    auto qbank = [&](int bank, int layer) { return qh + (bank * 2 + layer) * (H / 4); };
    float* h1c = st + H;
    float* maxima = st + 2 * H;

    // Encoder rows of a joint round's window (frames pf_base .. pf_base +
    // kWin - 1): loaded during the first barrier of a prediction update, when
    // the next round's frame is known, or directly by a round whose window
    // they are not.  pf_base = frame of candidate 0 (-1: none).
    uint32_t cand[kWin][KP];
    int pf_base = -1;
    bool do_pf = false;
    auto prefetch = [&]() {
#pragma unroll
        for (int d = 0; d < kWin; ++d) {
            const int f = pf_base + d;
            const bool ok = f < p.frames;
            const uint16_t* e = p.enc + (size_t)(ok ? f : 0) * p.enc_stride + 2 * lane;
#pragma unroll
            for (int j = 0; j < KP; ++j) cand[d][j] = ok ? *(const uint32_t*)(e + 128 * j) : 0u;
        }
    };

    // ---- grid barrier: publish this workgroup's word, wait for every tag ---------
    uint32_t epoch = 0;
    bool failed = false;
    auto barrier = [&](unsigned long long payload) -> unsigned long long {
        // this wave's state stores have completed before the word goes out
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const uint32_t tag = (epoch + 1) & 0x1fffu;
        unsigned long long* slot = words + (epoch & 1) * kDecMaxBlocks;
        if (tid == 0) __hip_atomic_store(slot + blk, payload | tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (do_pf) prefetch();  // in flight during the poll
        do_pf = false;
        unsigned long long mine = 0;
        uint32_t spins = 0;
        while (true) {
            bool ready = true;
            if (tid < nblocks) {
                mine = __hip_atomic_load(slot + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ready = ((uint32_t)mine & 0x1fffu) == tag;
            }
            if (__syncthreads_and(ready)) break;
            if ((++spins & 63) == 0) {
                // one thread decides, so the whole workgroup leaves together
                if (tid == 0)
                    stop_s = spins > kDecSpinLimit || __hip_atomic_load(&p.ws[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
                __syncthreads();
                if (stop_s) {
                    if (tid == 0) __hip_atomic_store(&p.ws[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    failed = true;
                    break;
                }
            }
            __builtin_amdgcn_s_sleep(1);
        }
        ++epoch;
        return mine;  // thread t holds workgroup t's word
    };
    // The joint rounds' barrier: thread c < kWin publishes this workgroup's key
    // for window frame c, each key tagged, so all go out together and the poll
    // itself gathers every workgroup's keys (thread t: workgroup t's, in got).
    // word-major ([parity][frame][workgroup]): the poll's lanes read consecutive words
    unsigned long long* wwords = (unsigned long long*)(p.ws + kDecState + 9 * H);  // [2][kWin][256]
    auto barrier_win = [&](unsigned long long key, unsigned long long (&got)[kWin]) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const uint32_t tag = (epoch + 1) & 0x1fffu;
        unsigned long long* slot = wwords + (size_t)(epoch & 1) * kDecMaxBlocks * kWin;
        if (tid < kWin) __hip_atomic_store(slot + tid * kDecMaxBlocks + blk, key | tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (do_pf) prefetch();
        do_pf = false;
        uint32_t spins = 0;
#pragma unroll
        for (int c = 0; c < kWin; ++c) got[c] = 0ull;
        while (true) {
            bool ready = true;
            if (tid < nblocks) {
#pragma unroll
                for (int c = 0; c < kWin; ++c) {
                    got[c] = __hip_atomic_load(slot + c * kDecMaxBlocks + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ready = ready && ((uint32_t)got[c] & 0x1fffu) == tag;
                }
            }
            if (__syncthreads_and(ready)) break;
            if ((++spins & 63) == 0) {
                if (tid == 0)
                    stop_s = spins > kDecSpinLimit || __hip_atomic_load(&p.ws[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
                __syncthreads();
                if (stop_s) {
                    if (tid == 0) __hip_atomic_store(&p.ws[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    failed = true;
                    break;
                }
            }
            __builtin_amdgcn_s_sleep(1);
        }
        ++epoch;
    };

    // long form: layer-0 recurrent sums of the candidate state [bank][H][4 gates]
    // (the committed bank is the other), published by the unit's owner
    int32_t* rs0w = (int32_t*)(p.ws + kDecState + 9 * H + kDecExtWords);

    // ---- weights into registers --------------------------------------------------
    const bool owns_unit = gw < H;
    const int u = owns_unit ? gw : 0;
    uint32_t wih[kLong ? 1 : 2][4][KP], whh[kLong ? 1 : 2][4][KP], wpj[KP];
    // long form: INT8 rows of W_hh0, W_hh1, W_ih1 and their scale / 127
    uint32_t qw[kLong ? 3 : 1][4][KD];
    float cq[3] = {1.0f, 1.0f, 1.0f};
    float bias[2][4];
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int g = 0; g < 4; ++g) bias[l][g] = p.b_ih[l][g * H + u] + p.b_hh[l][g * H + u];
    if constexpr (!kLong) {
#pragma unroll
        for (int l = 0; l < 2; ++l)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const size_t row = (size_t)(g * H + u) * H;
#pragma unroll
                for (int j = 0; j < KP; ++j) {
                    const int k = 2 * lane + 128 * j;
                    wih[l][g][j] = *(const uint32_t*)(p.w_ih[l] + row + k);
                    whh[l][g][j] = *(const uint32_t*)(p.w_hh[l] + row + k);
                }
            }
    } else {
        // decoder.cu:520-575: per-tensor maxima over the whole grid, scale =
        // max / 127 (1 for an all-zero matrix), q = quantize_i8(w / scale).
        const uint16_t* src[3] = {p.w_hh[0], p.w_hh[1], p.w_ih[1]};
        const size_t n8 = (size_t)H * H / 2;  // 16-byte chunks of a [4H x H] fp16 matrix
        const size_t gt = (size_t)blk * kDecThreads + tid, gs = (size_t)nblocks * kDecThreads;
        float mx[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            float a = 0.0f;
            for (size_t i = gt; i < n8; i += gs) {
                const uint4 v = ((const uint4*)src[m])[i];
                const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    a = __builtin_fmaxf(a, __builtin_fmaxf(__builtin_fabsf(lo16(w4[e])), __builtin_fabsf(hi16(w4[e]))));
            }
            mx[m] = wave_max(a);
        }
        if (lane == 0)
#pragma unroll
            for (int m = 0; m < 3; ++m) red_s[wave * 3 + m] = mx[m];
        __syncthreads();
        if (tid == 0)
#pragma unroll
            for (int m = 0; m < 3; ++m)
                st1(maxima + blk * 3 + m, __builtin_fmaxf(__builtin_fmaxf(red_s[m], red_s[3 + m]), __builtin_fmaxf(red_s[6 + m], red_s[9 + m])));
        barrier(0);
        float r[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            if (tid < nblocks) r[m] = ld1(maxima + tid * 3 + m);
            r[m] = wave_max(r[m]);
        }
        if (lane == 0)
#pragma unroll
            for (int m = 0; m < 3; ++m) red_s[wave * 3 + m] = r[m];
        __syncthreads();
        float scale[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const float t = __builtin_fmaxf(__builtin_fmaxf(red_s[m], red_s[3 + m]), __builtin_fmaxf(red_s[6 + m], red_s[9 + m]));
            scale[m] = t > 0.0f ? t / 127.0f : 1.0f;
            cq[m] = scale[m] / 127.0f;
        }
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int j = 0; j < KD; ++j) {
                    const int k = 4 * lane + 256 * j;
                    uint32_t word = 0;
                    if (k < H) {
                        const uint2 hv = *(const uint2*)(src[m] + (size_t)(g * H + u) * H + k);
                        word = (uint32_t)(uint8_t)quant_i8(lo16(hv.x) / scale[m]) | ((uint32_t)(uint8_t)quant_i8(hi16(hv.x) / scale[m]) << 8) |
                               ((uint32_t)(uint8_t)quant_i8(lo16(hv.y) / scale[m]) << 16) |
                               ((uint32_t)(uint8_t)quant_i8(hi16(hv.y) / scale[m]) << 24);
                    }
                    qw[m][g][j] = word;
                }
    }
#pragma unroll
    for (int j = 0; j < KP; ++j) wpj[j] = *(const uint32_t*)(p.w_proj + (size_t)u * H + 2 * lane + 128 * j);
    const float bpj = p.b_proj[u];
    uint32_t wj[2][KP];
    float wjs[2], wjb[2];
    int jid[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int i = 2 * gw + r;
        jid[r] = i < D ? T + i : (i < T + D ? i - D : -1);
        const int row = jid[r] < 0 ? p.outputs - 1 : jid[r];
#pragma unroll
        for (int j = 0; j < KP; ++j) {
            const int k = 2 * lane + 128 * j;
            if constexpr (kInt8) wj[r][j] = *(const uint16_t*)((const int8_t*)p.w_joint + (size_t)row * H + k);
            else wj[r][j] = *(const uint32_t*)((const uint16_t*)p.w_joint + (size_t)row * H + k);
        }
        wjs[r] = kInt8 ? p.joint_scales[row] : 1.0f;
        wjb[r] = p.b_joint[row];
    }

    // long form: layer 0 of every unit tid + 256 i is evaluated by this thread in
    // every workgroup (identical operations, so identical values everywhere):
    // its bias, committed / candidate cell state and the recurrent sums of the
    // state the next update consumes
    constexpr int NU = kLong ? (H + kDecThreads - 1) / kDecThreads : 1;
    float b0[NU][4], c0c[NU], c0n[NU];
    int r0[NU][4];
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        const int ui = min(tid + kDecThreads * i, H - 1);
        c0c[i] = c0n[i] = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            b0[i][g] = p.b_ih[0][g * H + ui] + p.b_hh[0][g * H + ui];
            r0[i][g] = 0;
        }
    }

    int frame = 0, symbols = 0, last = blank, count = 0, steps = 0, alt = 0;
    bool emitted = false, valid = false;
    float pv[2 * KP];
    // long form: integer recurrent sums [layer][gate] of the committed state
    // (rs) and of the candidate (rs_next); the owning wave's cell states
    int rs[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, rs_next[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
    float c_cur[2] = {0.0f, 0.0f}, c_new[2] = {0.0f, 0.0f};
    while (frame < p.frames && !failed) {
        if (!valid) {
            pf_base = frame;  // the next round's window loads during this update's first barrier
            do_pf = true;
            if constexpr (!kLong) {
                // ---- two LSTM layers on the last token's embedding (zeros before any)
#pragma unroll
                for (int l = 0; l < 2; ++l) {
                    if (owns_unit) {
                        float x[2 * KP], hv[2 * KP];
#pragma unroll
                        for (int j = 0; j < KP; ++j) {
                            const int k = 2 * lane + 128 * j;
                            if (l == 0) {
                                if (emitted) {
                                    const uint32_t e = *(const uint32_t*)(p.emb + (size_t)last * H + k);
                                    x[2 * j] = lo16(e);
                                    x[2 * j + 1] = hi16(e);
                                } else {
                                    x[2 * j] = x[2 * j + 1] = 0.0f;
                                }
                            } else {
                                const float2 v = ld2(hp(alt ^ 1, 0) + k);  // this update's layer-0 output
                                x[2 * j] = v.x;
                                x[2 * j + 1] = v.y;
                            }
                            const float2 hh = ld2(hp(alt, l) + k);
                            hv[2 * j] = hh.x;
                            hv[2 * j + 1] = hh.y;
                        }
                        float s[4];
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            float a = 0.0f;
#pragma unroll
                            for (int j = 0; j < KP; ++j) {
                                a = __builtin_fmaf(lo16(wih[l][g][j]), x[2 * j], a);
                                a = __builtin_fmaf(hi16(wih[l][g][j]), x[2 * j + 1], a);
                                a = __builtin_fmaf(lo16(whh[l][g][j]), hv[2 * j], a);
                                a = __builtin_fmaf(hi16(whh[l][g][j]), hv[2 * j + 1], a);
                            }
                            s[g] = wave_sum(a) + bias[l][g];
                        }
                        if (lane == 0) {
                            const float ig = sigmoid(s[0]), fg = sigmoid(s[1]), cg = tanhf(s[2]), og = sigmoid(s[3]);
                            const float cell = fg * ld1(cp(alt, l) + u) + ig * cg;
                            st1(cp(alt ^ 1, l) + u, cell);
                            st1(hp(alt ^ 1, l) + u, og * tanhf(cell));
                        }
                    }
                    barrier(0);
                    if (failed) break;
                }
                if (failed) break;
                // ---- projection of the new layer-1 output
                if (owns_unit) {
                    float a = 0.0f;
#pragma unroll
                    for (int j = 0; j < KP; ++j) {
                        const float2 v = ld2(hp(alt ^ 1, 1) + 2 * lane + 128 * j);
                        a = __builtin_fmaf(lo16(wpj[j]), v.x, a);
                        a = __builtin_fmaf(hi16(wpj[j]), v.y, a);
                    }
                    a = wave_sum(a) + bpj;
                    if (lane == 0) st1(pred + u, a);
                }
            } else {
                // ---- layer 0 of every unit, in every workgroup: recurrent sums of the
                // committed state + bias + the token's table row (decoder.cu:619-648)
#pragma unroll
                for (int i = 0; i < NU; ++i) {
                    const int ui = tid + kDecThreads * i;
                    if (ui < H) {
                        float s[4];
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const float tv = emitted ? h2f(p.table[(size_t)last * 4 * H + g * H + ui]) : 0.0f;
                            s[g] = __builtin_fmaf((float)r0[i][g], cq[0], b0[i][g]) + tv;
                        }
                        float h;
                        lstm_cell(s, c0c[i], c0n[i], h);
                        ((uint8_t*)q0_s)[ui] = (uint8_t)quant_i8(h * 127.0f);
                    }
                }
                __syncthreads();
                // ---- layer 1: its recurrent sums + W_ih1 x the new INT8 layer-0
                // output (decoder.cu:650-670); the layer-0 recurrent sums of the new
                // candidate state go out for the update after it is committed
                if (owns_unit) {
                    uint32_t x[KD];
#pragma unroll
                    for (int j = 0; j < KD; ++j) x[j] = 4 * lane + 256 * j < H ? q0_s[lane + 64 * j] : 0u;
                    int in[4], r0n[4];
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        int a = 0, d = 0;
#pragma unroll
                        for (int j = 0; j < KD; ++j) {
                            a = __builtin_amdgcn_sdot4((int)qw[2][g][j], (int)x[j], a, false);
                            d = __builtin_amdgcn_sdot4((int)qw[0][g][j], (int)x[j], d, false);
                        }
                        in[g] = a;
                        r0n[g] = d;
                    }
#pragma unroll
                    for (int off = 1; off < 64; off <<= 1)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            in[g] = add_level(in[g], off);
                            r0n[g] = add_level(r0n[g], off);
                        }
                    if (lane < 4) st_word((uint32_t*)rs0w + ((alt ^ 1) * H + u) * 4 + lane, (uint32_t)r0n[lane]);
                    if (lane == 0) {
                        float s[4];
#pragma unroll
                        for (int g = 0; g < 4; ++g)
                            s[g] = __builtin_fmaf((float)in[g], cq[2], __builtin_fmaf((float)rs[1][g], cq[1], bias[1][g]));
                        float h;
                        lstm_cell(s, c_cur[1], c_new[1], h);
                        st1(h1c + u, h);
                        qb_s[wave] = (uint32_t)(uint8_t)quant_i8(h * 127.0f);
                    }
                }
                __syncthreads();
                if (tid == 0 && 4 * blk < H)
                    st_word(qbank(alt ^ 1, 1) + blk, qb_s[0] | (qb_s[1] << 8) | (qb_s[2] << 16) | (qb_s[3] << 24));
                barrier(0);
                if (failed) break;
                // ---- projection of the new layer-1 output, and the layer-1 recurrent
                // sums of this candidate state for the update after it is committed
                if (owns_unit) {
                    uint32_t xq[KD];
#pragma unroll
                    for (int j = 0; j < KD; ++j) xq[j] = 4 * lane + 256 * j < H ? ld_word(qbank(alt ^ 1, 1) + lane + 64 * j) : 0u;
                    float a = 0.0f;
#pragma unroll
                    for (int j = 0; j < KP; ++j) {
                        const float2 v = ld2(h1c + 2 * lane + 128 * j);
                        a = __builtin_fmaf(lo16(wpj[j]), v.x, a);
                        a = __builtin_fmaf(hi16(wpj[j]), v.y, a);
                    }
                    a = wave_sum(a) + bpj;
                    if (lane == 0) st1(pred + u, a);
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        int d = 0;
#pragma unroll
                        for (int j = 0; j < KD; ++j) d = __builtin_amdgcn_sdot4((int)qw[1][g][j], (int)xq[j], d, false);
                        rs_next[1][g] = wave_isum(d);
                    }
                }
                // the candidate's layer-0 sums (published before the last barrier),
                // consumed by the next update once a token commits this state
#pragma unroll
                for (int i = 0; i < NU; ++i) {
                    const int ui = tid + kDecThreads * i;
                    if (ui < H)
#pragma unroll
                        for (int g = 0; g < 4; ++g) r0[i][g] = (int)ld_word((const uint32_t*)rs0w + ((alt ^ 1) * H + ui) * 4 + g);
                }
            }
            barrier(0);
            if (failed) break;
#pragma unroll
            for (int j = 0; j < KP; ++j) {
                const float2 v = ld2(pred + 2 * lane + 128 * j);
                pv[2 * j] = v.x;
                pv[2 * j + 1] = v.y;
            }
            valid = true;
        }
        // ---- joint round: frames frame .. frame + kWin - 1 against this prediction
        if (pf_base != frame) {
            pf_base = frame;
            prefetch();
        }
        {
            // the 2 x kWin dot products first, then their wave sums level by
            // level, so every butterfly step issues 2 kWin independent shuffles
            float acc[kWin][2];
#pragma unroll
            for (int c = 0; c < kWin; ++c) {
                float x[2 * KP];
#pragma unroll
                for (int j = 0; j < KP; ++j) {
                    const uint32_t ev = cand[c][j];
                    x[2 * j] = __builtin_fmaxf(lo16(ev) + pv[2 * j], 0.0f);
                    x[2 * j + 1] = __builtin_fmaxf(hi16(ev) + pv[2 * j + 1], 0.0f);
                }
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    float a = 0.0f;
#pragma unroll
                    for (int j = 0; j < KP; ++j) {
                        float w0, w1;
                        if constexpr (kInt8) {
                            w0 = (float)(int8_t)(wj[r][j] & 0xffu);
                            w1 = (float)(int8_t)((wj[r][j] >> 8) & 0xffu);
                        } else {
                            w0 = lo16(wj[r][j]);
                            w1 = hi16(wj[r][j]);
                        }
                        a = __builtin_fmaf(w0, x[2 * j], a);
                        a = __builtin_fmaf(w1, x[2 * j + 1], a);
                    }
                    acc[c][r] = a;
                }
            }
#pragma unroll
            for (int off = 1; off < 64; off <<= 1)
#pragma unroll
                for (int c = 0; c < kWin; ++c)
#pragma unroll
                    for (int r = 0; r < 2; ++r) acc[c][r] = add_level(acc[c][r], off);
#pragma unroll
            for (int c = 0; c < kWin; ++c) {
                float bs = -__builtin_huge_valf();
                int bi = 0x7fffffff;
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const float score = __builtin_fmaf(wjs[r], acc[c][r], wjb[r]);
                    const int id = jid[r];
                    if (id >= T) {
                        if (lane == 0) dur_sc[c][id - T] = score;  // workgroup 0 only
                    } else if (id >= 0) {
                        if (score > bs || (score == bs && id < bi)) {
                            bs = score;
                            bi = id;
                        }
                    }
                }
                if (lane == 0)
                    win_w[wave][c] = bi == 0x7fffffff ? 0ull
                                                      : (((unsigned long long)key_bits(bs) << 32) |
                                                         ((unsigned long long)(0xffffu - (uint32_t)bi) << 16));
            }
        }
        __syncthreads();
        // thread c: this workgroup's key for window frame c (workgroup 0's with
        // the first maximum of that frame's duration scores)
        unsigned long long key = 0ull;
        if (tid < kWin) {
            key = win_w[0][tid];
            for (int i = 1; i < 4; ++i) key = win_w[i][tid] > key ? win_w[i][tid] : key;
            if (blk == 0) {
                int d = 0;
                for (int i = 1; i < D; ++i)
                    if (dur_sc[tid][i] > dur_sc[tid][d]) d = i;
                key |= (unsigned long long)d << 13;
            }
        }
        // a blank run that leaves the window usually lands on its next frame:
        // that window loads during the barrier (a token's update reloads)
        pf_base = frame + kWin;
        do_pf = true;
        unsigned long long mine[kWin];
        barrier_win(key, mine);
        if (failed) break;
        // decisions of the window: per frame the largest key over the
        // workgroups is the best token; workgroup 0's carries the duration
        {
            if (tid == 0)
#pragma unroll
                for (int c = 0; c < kWin; ++c) win_dur[c] = (int)(((uint32_t)mine[c] >> 13) & 7u);
#pragma unroll
            for (int off = 1; off < 64; off <<= 1)
#pragma unroll
                for (int c = 0; c < kWin; ++c) {
                    mine[c] = max_level(mine[c], off);
                }
            if (lane == 0)
#pragma unroll
                for (int c = 0; c < kWin; ++c) win_w[wave][c] = mine[c];
            __syncthreads();
            if (tid < kWin) {
                unsigned long long b = win_w[0][tid];
                for (int i = 1; i < 4; ++i) b = win_w[i][tid] > b ? win_w[i][tid] : b;
                win_tok[tid] = key_token((uint32_t)b);
            }
            __syncthreads();
            // the greedy rules (decoder.cu:773-783) over the window, identical in
            // every thread: blank decisions keep the prediction, so later frames'
            // decisions in the window stand until a token or the window's end
            const int f0 = frame;
            int c = 0;
            while (true) {
                const int token = win_tok[c], dur = win_dur[c];
                ++steps;
                if (token != blank) {
                    if (blk == 0 && tid == 0 && count < p.capacity) p.tokens[count] = token;
                    ++count;
                    last = token;
                    emitted = true;
                    valid = false;
                    alt ^= 1;  // the candidate state becomes the committed one
                    if constexpr (kLong) {
                        c_cur[1] = c_new[1];
#pragma unroll
                        for (int g = 0; g < 4; ++g) rs[1][g] = rs_next[1][g];
#pragma unroll
                        for (int i = 0; i < NU; ++i) c0c[i] = c0n[i];
                    }
                }
                ++symbols;
                frame += dur;
                if (dur != 0 || symbols == p.max_symbols) {
                    if (dur == 0) ++frame;
                    symbols = 0;
                }
                if (token != blank || frame >= p.frames) break;
                c = frame - f0;
                if (c >= kWin) break;
            }
            __syncthreads();  // win_w / win_tok / win_dur are reused next round
        }
    }
    if (blk == 0 && tid == 0) {
        p.result[0] = count;
        p.result[1] = frame;
        p.result[2] = failed ? -2 : 0;
        p.result[3] = steps;
    }
}

// ---- the model's decoder width: 64 workgroups ------------------------------------
//
// At H = 640 the decode is a chain of small exchanges, not of arithmetic: every
// emitted token needs the layer-1 output, the prediction and the joint's best
// keys from all workgroups in turn.  Measured on an MI355X, one exchange (publish,
// poll until everybody's words are there) takes 2.74 us among 160 workgroups,
// 1.65 among 128, 1.31 among 64 and 1.13 among 16, on one XCD or on eight; but
// 3.3 us among 64 when every wave stores its own word instead of one wave a
// workgroup's ten in one 80-byte store, 3.7 with a second small store beside it.
// So this form uses 64 workgroups of ten waves (one hidden unit a wave, as above):
//  - What the others need travels in the exchange itself: a published word is
//    {fp32 value, epoch tag}, one contiguous store per workgroup, and thread t
//    of every workgroup polls word t, so there is no store-then-flag wait and no
//    load after the exchange.
//  - x = relu(enc + pred) of the window's frames is formed once per workgroup,
//    by thread k for feature k, and shared through LDS; a wave then scores four
//    joint rows against four frames (eight waves: 16 rows x 8 frames), rows
//    past 1024 go one to a workgroup and their eight frames to waves 8 and 9.
//  - An eleventh wave keeps the next 32 encoder rows in LDS, so that no poll
//    waits behind a load from HBM, and stores the layer-0 sums.
//  - Sums over the wave's 64 lanes keep the association of add_level's levels
//    1, 2, 4, ..., 32, but N sums reduced together halve their number at each
//    level (lanes_sum): 16 sums take about 60 instructions instead of 200.
// Every sum has the association of tdt_decode_kernel's, so the tokens are the same.
// 7500 frames, INT8 joint, long form: 41.1 -> 19.6 ms; on a slower box 69.3 ->
// 31.7 ms.  93 frames, fp16 form: 1003 -> 600 us on the latter.  Where a token's
// time goes (long form, 7500 frames, 2513 updates and 2520 joint rounds in 21.1
// ms, 8.4 us each, by cycle stamps in workgroup 0, which cost 2 % of it): layer
// 0 with the wait for its sums 1.5 us, layer 1 0.4 and its exchange 2.0, the
// projection 0.2 and its exchange 0.9, the joint 1.6 and its exchange 1.5, the
// greedy rules 0.3.  An exchange ends with the slowest workgroup, hence more than
// the 1.31 us it takes by itself, or less where work runs under it.
constexpr int k640H = 640, k640KP = 5, k640Blocks = 64, k640Waves = 10, k640Rows = 16;
constexpr int k640Threads = 64 * (k640Waves + 1);  // and a wave that loads the encoder rows
constexpr int k640Ring = 32;                        // encoder rows kept in LDS
static_assert(k640Ring >= kWin + kWin - 1 + 7, "the next round's window is loaded before its round");
constexpr int k640Outputs = k640Blocks * (k640Rows + 1);
// u32 offsets in the workspace, around the prediction at kDecState + 8 H
constexpr int k640Joint = 8;                                         // u64 [2][64][kWin]
constexpr int k640Max = k640Joint + 2 * kWin * k640Blocks * 2;     // u64 [64][3]
constexpr int k640Pred = k640Max + k640Blocks * 3 * 2;             // u64 [2][H]
constexpr int k640Out = kDecState + 8 * k640H;                      // float [H]: the last prediction
constexpr int k640H1 = k640Out + k640H;                            // u64 [2][H]
constexpr int k640H0 = k640H1 + 4 * k640H;                         // u64 [2][H] (fp16 form)
constexpr int k640R0 = k640H0 + 4 * k640H;                         // u64 [H][4] (long form)
static_assert(k640Pred + 4 * k640H <= k640Out, "workspace layout");
static_assert(k640R0 + 8 * k640H <= kDecState + 9 * k640H + kDecExtWords + 8 * k640H, "workspace size");

// 4 bytes global -> LDS per lane: lane l writes LDS bytes [lds_addr + 4 l, + 4).
// lds_addr must be wave-uniform; one wait state between the M0 write and the
// load that reads it.
__device__ __forceinline__ void dma4(const void* src, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src),
                 "s"(__builtin_amdgcn_readfirstlane(lds_addr))
                 : "memory", "m0");
}

// v[l ^ 4] and v[l ^ 8] of a row of 16 lanes, whatever the lanes hold.
__device__ __forceinline__ float xor4(float v) {
    const int s = __float_as_int(v);
    const int t = __builtin_amdgcn_update_dpp(s, s, 0x104, 0xf, 0x5, false);            // row_shl:4 into quads 0 and 2
    return __int_as_float(__builtin_amdgcn_update_dpp(t, s, 0x114, 0xf, 0xa, false));   // row_shr:4 into quads 1 and 3
}
__device__ __forceinline__ float xor8(float v) { return dpp_f<0x128>(v); }  // row_ror:8

// Wave sums of N values (4 or 16), lane l receiving that of value l mod N: at
// the first log2(N) levels the two lanes of a pair each keep one of two values
// and hand the other over.  Every sum is that of add_level's levels 1 .. 32.
template <int N> __device__ __forceinline__ float lanes_sum(float (&v)[N], int lane) {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        const bool b = lane & 1;
        v[i] = (b ? v[2 * i + 1] : v[2 * i]) + dpp_f<0xB1>(b ? v[2 * i] : v[2 * i + 1]);
    }
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {
        const bool b = lane & 2;
        v[i] = (b ? v[2 * i + 1] : v[2 * i]) + dpp_f<0x4E>(b ? v[2 * i] : v[2 * i + 1]);
    }
    float s;
    if constexpr (N == 16) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bool b = lane & 4;
            v[i] = (b ? v[2 * i + 1] : v[2 * i]) + xor4(b ? v[2 * i] : v[2 * i + 1]);
        }
        const bool b = lane & 8;
        s = (b ? v[1] : v[0]) + xor8(b ? v[0] : v[1]);
    } else {
        s = v[0] + xor4(v[0]);
        s = s + xor8(s);
    }
    return add_level(add_level(s, 16), 32);
}

// Integer wave sums (exact in any order).  Four values: lane l receives value
// 2 (l / 32) + (l / 16) % 2.
__device__ __forceinline__ int swap_add32(int a, int b) {  // lanes < 32: a's sums over l, l ^ 32; the others b's
    const auto q = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    return (int)q[0] + (int)q[1];
}
__device__ __forceinline__ int swap_add16(int a, int b) {  // even rows of 16: a's sums over l, l ^ 16; odd rows b's
    const auto q = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    return (int)q[0] + (int)q[1];
}
__device__ __forceinline__ int row_isum4(const int (&v)[4]) { return swap_add16(swap_add32(v[0], v[2]), swap_add32(v[1], v[3])); }
__device__ __forceinline__ int half_row_isum(int s) { return add_level(add_level(add_level(s, 1), 2), 4); }

// The greedy rules (decoder.cu:773-783) over a round's window, from its
// decisions (token | duration << 16 in lanes 0 .. kWin - 1): blank decisions
// keep the prediction, so later frames' decisions in the window stand until a
// token or the window's end.  emit(token) is called for a token.
struct GreedyState {
    int frame = 0, symbols = 0, steps = 0;
};
template <typename Emit>
__device__ __forceinline__ void greedy_round(GreedyState& g, int decided, int blank, int frames, int max_symbols, Emit&& emit) {
    const int f0 = g.frame;
    int c = 0;
    while (true) {
        const int d = __builtin_amdgcn_readlane(decided, c);
        const int token = d & 0xffff, dur = d >> 16;
        ++g.steps;
        if (token != blank) emit(token);
        ++g.symbols;
        g.frame += dur;
        if (dur != 0 || g.symbols == max_symbols) {
            if (dur == 0) ++g.frame;
            g.symbols = 0;
        }
        if (token != blank || g.frame >= frames) return;
        c = g.frame - f0;
        if (c >= kWin) return;
    }
}

template <bool kInt8, bool kLong>
__global__ __launch_bounds__(k640Threads) void tdt_decode_640_kernel(DecodeArgs p) {
    constexpr int H = k640H, KP = k640KP, KD = 3, NB = k640Blocks;
    typedef unsigned long long u64;
    __shared__ __attribute__((aligned(16))) uint16_t enc_s[k640Ring][H];  // encoder rows frame .. frame + k640Ring - 1
    __shared__ float x_s[kWin][H];                       // relu(enc + pred) of the window's frames
    __shared__ float h_s[kLong ? 1 : 4][H];              // long: layer 1's output; fp16: [bank][layer]
    __shared__ uint32_t q_s[2][kLong ? H / 4 : 1];       // long: the INT8 outputs of layers 0 and 1
    __shared__ u64 key_s[kWin][8];                       // best key of four rows each, entry 4: of the row past 1024
    __shared__ __attribute__((aligned(16))) float dur_s[kWin][8];
    __shared__ u64 win_s[8][kWin];                       // best key of the eight workgroups a wave polled
    __shared__ float out_s[2][k640Waves];               // this workgroup's values of an exchange
    __shared__ int r0_s[kLong ? k640Waves * 4 : 1];     // and its layer-0 sums
    __shared__ int win_dur[kWin];
    __shared__ float red_s[k640Waves * 3];
    __shared__ int stop_s;
    const int blk = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int u = min(blk * k640Waves + wave, H - 1);  // this wave's hidden unit
    const int T = p.token_outputs, D = p.durations, blank = T - 1;
    auto words = [&](int off) { return (u64*)(p.ws + off); };

    if (tid == 0) stop_s = 0;
    if (tid < kWin * 8) {
        key_s[tid >> 3][tid & 7] = 0ull;
        dur_s[tid >> 3][tid & 7] = 0.0f;
    }
    __syncthreads();

    auto publish = [&](u64* w, uint32_t v, uint32_t tag) {
        __hip_atomic_store(w, ((u64)v << 32) | tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // the workgroup's ten values, gathered in out_s[i], to their words
    auto publish_out = [&](u64* w, int i, uint32_t tag) {
        __syncthreads();
        if (wave == 0 && lane < k640Waves) publish(w + blk * k640Waves + lane, __float_as_uint(out_s[i][lane]), tag);
    };
    // The wave polls its lanes' words until all carry the tag.  Bounded: after
    // kDecSpinLimit polls, or once another workgroup gave up, the wave sets
    // stop_s, which the workgroup checks behind its next barrier.
    auto poll = [&](const u64* w, uint32_t mask, uint32_t tag) -> u64 {
        u64 v;
        uint32_t spins = 0;
        while (true) {
            v = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__builtin_amdgcn_ballot_w64(((uint32_t)v & mask) != tag) == 0) break;
            if ((++spins & 63) == 0 && (spins > kDecSpinLimit || ld_word(&p.ws[0]) != 0u)) {
                st_word(&p.ws[0], 1u);
                stop_s = 1;
                break;
            }
        }
        return v;
    };
    // Four words a lane at once, with the tag the first poll usually finds.
    auto poll4 = [&](const u64* w, uint32_t tag, int (&v)[4]) {
        u64 q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = __hip_atomic_load(w + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (__builtin_amdgcn_ballot_w64((uint32_t)q[i] != tag) != 0) q[i] = poll(w + i, 0xffffffffu, tag);
            v[i] = (int)(q[i] >> 32);
        }
    };
    auto value = [](u64 w) { return __uint_as_float((uint32_t)(w >> 32)); };

    // The round's decisions from the waves' keys, in every wave: lanes c, c + 8,
    // ... hold window frame c's, token | duration << 16.  The largest key is the
    // best token; workgroup 0's carries the duration.
    auto max8 = [](u64 v) {  // over lanes l, l ^ 8, l ^ 16, ...
        const u64 o = ((u64)(uint32_t)dpp_mov<0x128>((int)(v >> 32)) << 32) | (uint32_t)dpp_mov<0x128>((int)(uint32_t)v);
        return max_level(max_level(o > v ? o : v, 16), 32);
    };
    auto decisions = [&]() {
        const u64 b = max8(win_s[lane >> 3][lane & 7]);
        return key_token((uint32_t)b) | (win_dur[lane & 7] << 16);
    };

    // ---- wave 10: the encoder rows ---------------------------------------------
    // It follows the decisions and keeps the ring full with direct-to-LDS loads,
    // a round ahead of their use (a round advances at most kWin - 1 + 7 frames),
    // so that no exchange waits behind a load from HBM.  It meets every barrier
    // of the other waves (their loop below): at the start, and per update and
    // per round.
    if (wave == k640Waves) {
        const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)&enc_s[0][0];
        int loaded = 0;
        auto load_to = [&](int end) {
            for (; loaded < min(end, p.frames); ++loaded)
#pragma unroll
                for (int j = 0; j < KP; ++j)
                    dma4(p.enc + (size_t)loaded * p.enc_stride + 2 * lane + 128 * j,
                         ring + (uint32_t)(loaded & (k640Ring - 1)) * (2 * H) + 256 * j);
        };
        load_to(k640Ring);
        if constexpr (kLong) __syncthreads();  // the maxima
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        GreedyState g;
        bool valid = false;
        uint32_t updates = 0;
        while (g.frame < p.frames) {
            if (!valid) {
                ++updates;
                __syncthreads();
                __syncthreads();
                if constexpr (!kLong) {
                    if (stop_s) return;
                    __syncthreads();
                }
                __syncthreads();
                if (stop_s) return;
                // one bank of layer-0 sums: every workgroup has taken part in the
                // layer-1 exchange just polled, so it has read the last update's
                if constexpr (kLong)
                    if (lane < 4 * k640Waves)
                        publish(words(k640R0) + blk * (4 * k640Waves) + lane, (uint32_t)r0_s[lane], updates);
                __syncthreads();
                valid = true;
            }
            __syncthreads();
            if (stop_s) return;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            __syncthreads();
            if (stop_s) return;
            greedy_round(g, decisions(), blank, p.frames, p.max_symbols, [&](int) { valid = false; });
            load_to(g.frame + k640Ring);
        }
        return;
    }

    // ---- weights into registers ------------------------------------------------
    uint32_t wih[kLong ? 1 : 2][4][KP], whh[kLong ? 1 : 2][4][KP], wpj[KP];
    uint32_t qw[kLong ? 3 : 1][4][KD];  // long form: INT8 rows of W_hh0, W_hh1, W_ih1
    float cq[3] = {1.0f, 1.0f, 1.0f};   // and their scale / 127
    // the gate whose sum this lane holds after a reduction, and its bias
    const int gate = kLong ? lane >> 4 : lane & 3;
    const float bias1 = p.b_ih[1][gate * H + u] + p.b_hh[1][gate * H + u];
    const float bias0 = p.b_ih[0][gate * H + u] + p.b_hh[0][gate * H + u];
    if constexpr (!kLong) {
#pragma unroll
        for (int l = 0; l < 2; ++l)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const size_t row = (size_t)(g * H + u) * H + 2 * lane;
#pragma unroll
                for (int j = 0; j < KP; ++j) {
                    wih[l][g][j] = *(const uint32_t*)(p.w_ih[l] + row + 128 * j);
                    whh[l][g][j] = *(const uint32_t*)(p.w_hh[l] + row + 128 * j);
                }
            }
        for (int i = tid; i < 4 * H; i += H) (&h_s[0][0])[i] = 0.0f;
    } else {
        // per-tensor maxima over the whole grid, as above
        const uint16_t* src[3] = {p.w_hh[0], p.w_hh[1], p.w_ih[1]};
        constexpr int n8 = H * H / 2;  // 16-byte chunks of a [4H x H] fp16 matrix
        float mx[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            float a = 0.0f;
            for (int i = blk * H + tid; i < n8; i += NB * H) {
                const uint4 v = ((const uint4*)src[m])[i];
                const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    a = __builtin_fmaxf(a, __builtin_fmaxf(__builtin_fabsf(lo16(w4[e])), __builtin_fabsf(hi16(w4[e]))));
            }
            mx[m] = wave_max(a);
        }
        if (lane == 0)
#pragma unroll
            for (int m = 0; m < 3; ++m) red_s[wave * 3 + m] = mx[m];
        __syncthreads();
        if (tid < 3) {
            float a = red_s[tid];
            for (int i = 1; i < k640Waves; ++i) a = __builtin_fmaxf(a, red_s[i * 3 + tid]);
            publish(words(k640Max) + blk * 3 + tid, __float_as_uint(a), 1u);
        }
        float scale[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const float t = wave_max(value(poll(words(k640Max) + lane * 3 + m, 0xffffffffu, 1u)));
            scale[m] = t > 0.0f ? t / 127.0f : 1.0f;
            cq[m] = scale[m] / 127.0f;
        }
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int j = 0; j < KD; ++j) {
                    const int k = 4 * lane + 256 * j;
                    uint32_t word = 0;
                    if (k < H) {
                        const uint2 hv = *(const uint2*)(src[m] + (size_t)(g * H + u) * H + k);
                        word = (uint32_t)(uint8_t)quant_i8(lo16(hv.x) / scale[m]) | ((uint32_t)(uint8_t)quant_i8(hi16(hv.x) / scale[m]) << 8) |
                               ((uint32_t)(uint8_t)quant_i8(lo16(hv.y) / scale[m]) << 16) |
                               ((uint32_t)(uint8_t)quant_i8(hi16(hv.y) / scale[m]) << 24);
                    }
                    qw[m][g][j] = word;
                }
    }
#pragma unroll
    for (int j = 0; j < KP; ++j) wpj[j] = *(const uint32_t*)(p.w_proj + (size_t)u * H + 2 * lane + 128 * j);
    const float bpj = p.b_proj[u];
    // joint rows: waves 0 .. 7 own rows 4 (wave % 4) .. + 3 of the workgroup's 16
    // for frames 4 (wave / 4) .. + 3 of the window, waves 8 and 9 the row past
    // 1024 if there is one.  Logical order: the duration rows first, so
    // workgroup 0 holds them all.
    const bool extra = wave >= 8;
    const int fh = extra ? wave - 8 : wave >> 2;
    auto joint_id = [&](int r) {
        const int i = extra ? (r == 0 ? NB * k640Rows + blk : T + D) : blk * k640Rows + 4 * (wave & 3) + r;
        return i < D ? T + i : (i < T + D ? i - D : -1);
    };
    // The long form keeps INT8 weights as fp32 values, the fp16 form, short of
    // registers, four to a dword; fp16 weights stay pairs.
    constexpr bool kWide = kInt8 && kLong;
    constexpr int JW = kWide ? 2 * KP : (kInt8 ? (KP + 1) / 2 : KP);
    uint32_t wj[4][JW];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int id = joint_id(r), row = id < 0 ? p.outputs - 1 : id;
#pragma unroll
        for (int j = 0; j < KP; ++j) {
            const size_t at = (size_t)row * H + 2 * lane + 128 * j;
            if constexpr (kInt8) {
                const uint32_t w = *(const uint16_t*)((const int8_t*)p.w_joint + at);
                if constexpr (kWide) {
                    wj[r][2 * j] = __float_as_uint((float)(int8_t)(w & 0xffu));
                    wj[r][2 * j + 1] = __float_as_uint((float)(int8_t)((w >> 8) & 0xffu));
                } else {
                    wj[r][j / 2] = (j & 1) ? wj[r][j / 2] | (w << 16) : w;
                }
            } else {
                wj[r][j] = *(const uint32_t*)((const uint16_t*)p.w_joint + at);
            }
        }
    }
    // the row whose sums this lane holds after a reduction
    const int my_id = joint_id(extra ? 0 : lane & 3);
    const int my_row = my_id < 0 ? p.outputs - 1 : my_id;
    const float my_scale = kInt8 ? p.joint_scales[my_row] : 1.0f, my_bias = p.b_joint[my_row];

    // long form: thread t evaluates layer 0 of unit t in every workgroup
    float b0[4], c0c = 0.0f, c0n = 0.0f;
#pragma unroll
    for (int g = 0; g < 4; ++g) b0[g] = kLong ? p.b_ih[0][g * H + tid] + p.b_hh[0][g * H + tid] : 0.0f;

    __syncthreads();
    GreedyState g;
    int last = blank, count = 0, alt = 0;
    uint32_t updates = 0, rounds = 0;
    bool emitted = false, valid = false, failed = false;
    float pv = 0.0f;                                                // prediction value of feature tid
    int rs = 0, rs_next = 0;                                        // long: layer 1's recurrent sum of this lane's gate
    float c_cur[2] = {0.0f, 0.0f}, c_new[2] = {0.0f, 0.0f};         // cell states of unit u
    while (g.frame < p.frames) {
        // Packed weights are unpacked where they are used: without this the
        // compiler hoists the conversions out of the loop and spills.  The
        // fp16 form still spills a few of the 168 registers that eleven waves
        // leave (6 with an INT8 joint, 9 with an fp16 one); the long form none.
        auto keep = [](uint32_t& w) { asm volatile("" : "+v"(w)); };
#pragma unroll
        for (int j = 0; j < KP; ++j) {
            keep(wpj[j]);
            if constexpr (!kLong)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    keep(wih[i >> 2][i & 3][j]);
                    keep(whh[i >> 2][i & 3][j]);
                }
        }
        if constexpr (!kWide)
#pragma unroll
            for (int i = 0; i < 4 * JW; ++i) keep(wj[i / JW][i % JW]);
        if (!valid) {
            const uint32_t tag = ++updates;
            const int par = (int)(tag & 1u);
            u64* h1w = words(k640H1) + par * H;
            u64* pw = words(k640Pred) + par * H;
            if constexpr (!kLong) {
                // ---- two LSTM layers on the last token's embedding (zeros before any)
                u64* h0w = words(k640H0) + par * H;
#pragma unroll
                for (int l = 0; l < 2; ++l) {
                    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int j = 0; j < KP; ++j) {
                        const int k = 2 * lane + 128 * j;
                        float2 x = make_float2(0.0f, 0.0f);
                        if (l == 0) {
                            if (emitted) {
                                const uint32_t e = *(const uint32_t*)(p.emb + (size_t)last * H + k);
                                x = make_float2(lo16(e), hi16(e));
                            }
                        } else {
                            x = *(const float2*)&h_s[(alt ^ 1) * 2][k];  // this update's layer-0 output
                        }
                        const float2 hv = *(const float2*)&h_s[alt * 2 + l][k];
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            s[g] = __builtin_fmaf(lo16(wih[l][g][j]), x.x, s[g]);
                            s[g] = __builtin_fmaf(hi16(wih[l][g][j]), x.y, s[g]);
                            s[g] = __builtin_fmaf(lo16(whh[l][g][j]), hv.x, s[g]);
                            s[g] = __builtin_fmaf(hi16(whh[l][g][j]), hv.y, s[g]);
                        }
                    }
                    const float v = lanes_sum(s, lane) + (l == 0 ? bias0 : bias1);
                    const int act = __float_as_int(gate == 2 ? tanhf(v) : sigmoid(v));
                    const float ig = __int_as_float(__builtin_amdgcn_readlane(act, 0)), fg = __int_as_float(__builtin_amdgcn_readlane(act, 1));
                    const float cg = __int_as_float(__builtin_amdgcn_readlane(act, 2)), og = __int_as_float(__builtin_amdgcn_readlane(act, 3));
                    c_new[l] = fg * c_cur[l] + ig * cg;
                    const float h = og * tanhf(c_new[l]);
                    u64* w = l == 0 ? h0w : h1w;
                    if (lane == 0) out_s[0][wave] = h;
                    publish_out(w, 0, tag);
                    h_s[(alt ^ 1) * 2 + l][tid] = value(poll(w + tid, 0xffffffffu, tag));
                    __syncthreads();
                    if (stop_s) failed = true;
                    if (failed) break;
                }
                if (failed) break;
            } else {
                // ---- layer 0 of unit tid: recurrent sums of the committed state +
                // bias + the token's table row (decoder.cu:619-648)
                float s[4];
                uint16_t tv[4] = {0, 0, 0, 0};
                int r0[4] = {0, 0, 0, 0};
                if (emitted) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) tv[g] = p.table[(size_t)last * 4 * H + g * H + tid];
                    // published by the last update after its layer-1 exchange; overwritten
                    // after this update's, which waits for this workgroup
                    poll4(words(k640R0) + tid * 4, tag - 1, r0);
                }
#pragma unroll
                for (int g = 0; g < 4; ++g) s[g] = __builtin_fmaf((float)r0[g], cq[0], b0[g]) + h2f(tv[g]);
                float h0;
                lstm_cell(s, c0c, c0n, h0);
                ((uint8_t*)q_s[0])[tid] = (uint8_t)quant_i8(h0 * 127.0f);
                __syncthreads();
                // ---- layer 1: its recurrent sums + W_ih1 x the new INT8 layer-0
                // output (decoder.cu:650-670), and the layer-0 recurrent sums of the
                // new candidate state, which go out for the update after it is committed
                uint32_t x[KD];
#pragma unroll
                for (int j = 0; j < KD; ++j) x[j] = 4 * lane + 256 * j < H ? q_s[0][lane + 64 * j] : 0u;
                int in[4], r0n[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    int a = 0, d = 0;
#pragma unroll
                    for (int j = 0; j < KD; ++j) {
                        a = __builtin_amdgcn_sdot4((int)qw[2][g][j], (int)x[j], a, false);
                        d = __builtin_amdgcn_sdot4((int)qw[0][g][j], (int)x[j], d, false);
                    }
                    in[g] = a;
                    r0n[g] = d;
                }
                const int ia = row_isum4(in), ra = row_isum4(r0n);
                const bool hi = lane & 8;  // lanes 8 .. 15 of a row take the layer-0 sum, the others layer 1's
                const int sum = half_row_isum((hi ? ra : ia) + dpp_mov<0x128>(hi ? ia : ra));
                if ((lane & 15) == 8) r0_s[wave * 4 + gate] = sum;  // wave 10 publishes them
                const float v = __builtin_fmaf((float)sum, cq[2], __builtin_fmaf((float)rs, cq[1], bias1));
                const int act = __float_as_int(det_gate(v, gate == 2));
                const float ig = __int_as_float(__builtin_amdgcn_readlane(act, 0)), fg = __int_as_float(__builtin_amdgcn_readlane(act, 16));
                const float cg = __int_as_float(__builtin_amdgcn_readlane(act, 32)), og = __int_as_float(__builtin_amdgcn_readlane(act, 48));
                c_new[1] = __builtin_fmaf(fg, c_cur[1], ig * cg);
                const float hn = og * det_tanh(c_new[1]);
                if (lane == 0) out_s[0][wave] = hn;
                publish_out(h1w, 0, tag);
                const float h1 = value(poll(h1w + tid, 0xffffffffu, tag));
                h_s[0][tid] = h1;
                ((uint8_t*)q_s[1])[tid] = (uint8_t)quant_i8(h1 * 127.0f);
                __syncthreads();
                if (stop_s) {
                    failed = true;
                    break;
                }
            }
            // ---- projection of the new layer-1 output
            const float* h1 = kLong ? h_s[0] : h_s[(alt ^ 1) * 2 + 1];
            float a = 0.0f;
#pragma unroll
            for (int j = 0; j < KP; ++j) {
                const float2 v = *(const float2*)&h1[2 * lane + 128 * j];
                a = __builtin_fmaf(lo16(wpj[j]), v.x, a);
                a = __builtin_fmaf(hi16(wpj[j]), v.y, a);
            }
            a = wave_sum(a) + bpj;
            if (lane == 0) out_s[1][wave] = a;
            publish_out(pw, 1, tag);
            if constexpr (kLong) {
                // layer 1's recurrent sums of this candidate state, for the update after it is committed
                uint32_t x[KD];
#pragma unroll
                for (int j = 0; j < KD; ++j) x[j] = 4 * lane + 256 * j < H ? q_s[1][lane + 64 * j] : 0u;
                int d[4] = {0, 0, 0, 0};
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int j = 0; j < KD; ++j) d[g] = __builtin_amdgcn_sdot4((int)qw[1][g][j], (int)x[j], d[g], false);
                const int s = row_isum4(d);
                rs_next = half_row_isum(s + dpp_mov<0x128>(s));
            }
            pv = value(poll(pw + tid, 0xffffffffu, tag));
            valid = true;
        }
        // ---- joint round: frames frame .. frame + kWin - 1 against this prediction
#pragma unroll
        for (int c = 0; c < kWin; ++c) {
            const float e = g.frame + c < p.frames ? h2f(enc_s[(g.frame + c) & (k640Ring - 1)][tid]) : 0.0f;
            x_s[c][tid] = __builtin_fmaxf(e + pv, 0.0f);
        }
        __syncthreads();
        if (stop_s) {
            failed = true;
            break;
        }
        auto score_key = [&](float sum, float& score) -> u64 {
            score = __builtin_fmaf(my_scale, sum, my_bias);
            if (my_id < 0 || my_id >= T || score != score) return 0ull;
            return ((u64)key_bits(score) << 32) | ((u64)(0xffffu - (uint32_t)my_id) << 16);
        };
        auto wpair = [&](int r, int j, float& w0, float& w1) {
            if constexpr (kWide) {
                w0 = __uint_as_float(wj[r][2 * j]);
                w1 = __uint_as_float(wj[r][2 * j + 1]);
            } else if constexpr (kInt8) {
                w0 = (float)(int8_t)(wj[r][j / 2] >> (16 * (j & 1)));
                w1 = (float)(int8_t)(wj[r][j / 2] >> (16 * (j & 1) + 8));
            } else {
                w0 = lo16(wj[r][j]);
                w1 = hi16(wj[r][j]);
            }
        };
        if (!extra) {
            float acc[16];  // [frame][row]
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
            for (int j = 0; j < KP; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float2 x = *(const float2*)&x_s[4 * fh + c][2 * lane + 128 * j];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float w0, w1;
                        wpair(r, j, w0, w1);
                        acc[4 * c + r] = __builtin_fmaf(w0, x.x, acc[4 * c + r]);
                        acc[4 * c + r] = __builtin_fmaf(w1, x.y, acc[4 * c + r]);
                    }
                }
            float score;
            u64 key = score_key(lanes_sum(acc, lane), score);
            const int c = 4 * fh + ((lane >> 2) & 3);
            if (lane < 16 && my_id >= T) dur_s[c][my_id - T] = score;  // workgroup 0 only
            key = max_level(max_level(key, 1), 2);
            if (lane < 16 && (lane & 3) == 0) key_s[c][wave & 3] = key;
        } else if (my_id >= 0) {
            float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < KP; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float2 x = *(const float2*)&x_s[4 * fh + c][2 * lane + 128 * j];
                    float w0, w1;
                    wpair(0, j, w0, w1);
                    acc[c] = __builtin_fmaf(w0, x.x, acc[c]);
                    acc[c] = __builtin_fmaf(w1, x.y, acc[c]);
                }
            float score;
            const u64 key = score_key(lanes_sum(acc, lane), score);
            if (lane < 4) key_s[4 * fh + lane][4] = key;
        }
        __syncthreads();
        const uint32_t jtag = (rounds + 1) & 0x1fffu;
        u64* jw = words(k640Joint) + (rounds & 1u) * (kWin * NB);  // [workgroup][window frame]
        ++rounds;
        if (wave == 0) {
            // lanes 8 c .. 8 c + 7: the workgroup's key for window frame c
            // (workgroup 0's with the first maximum of its duration scores)
            const int c = lane >> 3;
            u64 key = key_s[c][lane & 7];
            key = max_level(max_level(max_level(key, 1), 2), 4);
            if (blk == 0) {
                float best = dur_s[c][0];
                int d = 0;
#pragma unroll
                for (int i = 1; i < 8; ++i)
                    if (i < D && dur_s[c][i] > best) {
                        best = dur_s[c][i];
                        d = i;
                    }
                key |= (u64)d << 13;
            }
            if ((lane & 7) == 0)
                __hip_atomic_store(jw + blk * kWin + c, key | jtag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (wave < 8) {
            // wave w: the keys of workgroups 8 w .. 8 w + 7
            const u64 b = poll(jw + tid, 0x1fffu, jtag);
            if (tid < kWin) win_dur[tid] = (int)((uint32_t)b >> 13) & 7;
            const u64 m = max8(b);
            if (lane < kWin) win_s[wave][lane] = m;
        }
        __syncthreads();
        if (stop_s) {
            failed = true;
            break;
        }
        // identical in every wave
        greedy_round(g, decisions(), blank, p.frames, p.max_symbols, [&](int token) {
            if (blk == 0 && tid == 0 && count < p.capacity) p.tokens[count] = token;
            ++count;
            last = token;
            emitted = true;
            valid = false;
            alt ^= 1;  // the candidate state becomes the committed one
            c_cur[0] = c_new[0];
            c_cur[1] = c_new[1];
            rs = rs_next;
            c0c = c0n;
        });
    }
    if (blk == 0) {
        ((float*)p.ws)[k640Out + tid] = pv;
        if (tid == 0) {
            p.result[0] = count;
            p.result[1] = g.frame;
            p.result[2] = failed ? -2 : 0;
            p.result[3] = g.steps;
        }
    }
}

__global__ void decode_clear_kernel(uint32_t* ws, int words) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += gridDim.x * blockDim.x) ws[i] = 0u;
}

}  // namespace

// fp16 form: h, c (2 banks x 2 layers) and the prediction; long form: INT8
// banks (H words), candidate layer-1 output (H), maxima (3 x blocks, <= 6H
// for H >= 128) and the prediction at the same offset 8H; after the joint
// rounds' words, the long form's layer-0 recurrent sums (2 banks x H x 4).
int decode_workspace_words(int hidden) { return kDecState + 9 * hidden + kDecExtWords + 8 * hidden; }

int launch_tdt_decode(const uint16_t* enc, int frames, int enc_stride, const uint16_t* emb, const uint16_t* table, const uint16_t* const* w_ih,
                      const uint16_t* const* w_hh, const float* const* b_ih, const float* const* b_hh, const uint16_t* w_proj,
                      const float* b_proj, const void* w_joint, int joint_int8, const float* joint_scales, const float* b_joint,
                      int hidden, int token_outputs, int durations, int max_symbols, int32_t* tokens, int capacity, int32_t* result,
                      uint32_t* workspace, hipStream_t s) {
    int blocks = cu_count();
    if (blocks > kDecMaxBlocks) blocks = kDecMaxBlocks;
    const int outputs = token_outputs + durations;
    if (hidden > 4 * blocks || outputs > 8 * blocks) {
        set_error("decode needs hidden <= %d and outputs <= %d on this GPU", 4 * blocks, 8 * blocks);
        return -1;
    }
    // only as many workgroups as own a hidden unit (4 each) or joint rows (8
    // each): every further one would only add a participant to each barrier
    const int needed = max((hidden + 3) / 4, (outputs + 7) / 8);
    if (needed < blocks) blocks = needed;
    if (hidden > 4 * blocks || outputs > 8 * blocks) {
        set_error("decode needs hidden <= %d and outputs <= %d on this GPU", 4 * blocks, 8 * blocks);
        return -1;
    }
    DecodeArgs a{};
    a.enc = enc;
    a.emb = emb;
    a.table = table;
    for (int l = 0; l < 2; ++l) {
        a.w_ih[l] = w_ih[l];
        a.w_hh[l] = w_hh[l];
        a.b_ih[l] = b_ih[l];
        a.b_hh[l] = b_hh[l];
    }
    a.w_proj = w_proj;
    a.b_proj = b_proj;
    a.w_joint = w_joint;
    a.joint_scales = joint_scales;
    a.b_joint = b_joint;
    a.tokens = tokens;
    a.result = result;
    a.ws = workspace;
    a.frames = frames;
    a.enc_stride = enc_stride;
    a.outputs = outputs;
    a.token_outputs = token_outputs;
    a.durations = durations;
    a.max_symbols = max_symbols;
    a.capacity = capacity;
    decode_clear_kernel<<<16, 256, 0, s>>>(workspace, decode_workspace_words(hidden));
    static_assert(k640H > 4 * k640Blocks, "a GPU that passes the check above holds the 640 kernel's workgroups too");
    if (hidden == k640H && outputs <= k640Outputs) {
        if (table) {
            if (joint_int8) tdt_decode_640_kernel<true, true><<<k640Blocks, k640Threads, 0, s>>>(a);
            else tdt_decode_640_kernel<false, true><<<k640Blocks, k640Threads, 0, s>>>(a);
        } else {
            if (joint_int8) tdt_decode_640_kernel<true, false><<<k640Blocks, k640Threads, 0, s>>>(a);
            else tdt_decode_640_kernel<false, false><<<k640Blocks, k640Threads, 0, s>>>(a);
        }
        return 0;
    }
    switch (hidden >> 7) {
#define PK_DEC_CASE(KP)                                                                          \
    case KP:                                                                                     \
        if (table) {                                                                             \
            if (joint_int8) tdt_decode_kernel<true, KP, true><<<blocks, kDecThreads, 0, s>>>(a);  \
            else tdt_decode_kernel<false, KP, true><<<blocks, kDecThreads, 0, s>>>(a);            \
        } else {                                                                                 \
            if (joint_int8) tdt_decode_kernel<true, KP, false><<<blocks, kDecThreads, 0, s>>>(a); \
            else tdt_decode_kernel<false, KP, false><<<blocks, kDecThreads, 0, s>>>(a);           \
        }                                                                                        \
        break;
        PK_DEC_CASE(1) PK_DEC_CASE(2) PK_DEC_CASE(3) PK_DEC_CASE(4) PK_DEC_CASE(5) PK_DEC_CASE(6) PK_DEC_CASE(7) PK_DEC_CASE(8)
#undef PK_DEC_CASE
    default: break;
    }
    return 0;
}

}  // namespace pk
