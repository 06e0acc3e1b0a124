// q8_attn.hip -- decoder support kernels around the Q8_0 matmuls, for the
// synthetic decoder and the decode graph (included by q8_kernels.hip, one code
// object):
//   q8_rope_append   rotary embedding of q and k, k and v narrowed to the f16
//                    KV cache                     (gpu.cu rope_append 525-581, ops.rs:152-166)
//   q8_attn_decode   one token against the cache, positions split over
//                    workgroups, combined by the last or by the next kernel
//                    (gpu.cu attention_split 649-733, combine 735-762)
//   q8_attn_prefill  causal attention of n tokens on f16 MFMA (split operands),
//                    online softmax               (compute.rs attend_host 1075-1126)
//   q8_synth         seeded synthetic Q8_0 blocks for the benchmark decoder
//   q8_advance       the position a captured step reads, moved on the device
//
// The position a step works at is read from device memory, so one captured
// graph replays at every position (model.rs:676-731, cuda/mod.rs position_ptr).
// Head width is Q8_ATTN_HEAD_DIM (64): the configuration these kernels serve.

// ---------------------------------------------------------------------------
// RoPE + KV append.  One thread per (token, head, dimension pair) over the q
// heads, then the k heads, then the v heads.  Pairs (2i, 2i+1) inside each head
// rotate by angle = position * freq[i] (pairs at or beyond n_rot/2 are
// copied), computed in f32 exactly as the reference writes it
// (x0*cos - x1*sin, x0*sin + x1*cos, no contraction).  freq[i] =
// base^(-2i/n_rot) comes from the host's powf, the function the reference's
// RopeTable calls (ops.rs:121-131): at position p an ulp of freq moves the
// angle by p ulps, so a device pow would drift from the reference's table by
// ~p * 6e-8 in cos and sin.  q is rotated in place;
// rotated k and plain v are rounded to f16 (nearest even) into the cache at
// rows position + t.  Rows at or past `capacity` are never written.
// ---------------------------------------------------------------------------

extern "C" __global__ __launch_bounds__(256) void q8_rope_append(Q8RopeArgs a) {
    const int start = *a.position;
    const int half = a.head_dim >> 1;
    const int kv_dim = a.n_kv * a.head_dim;
    const int heads = a.n_head + 2 * a.n_kv;
    const long long total = (long long)a.n * heads * half;
    for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (long long)gridDim.x * blockDim.x) {
        const int pair = (int)(idx % half);
        const long long th = idx / half;
        const int hh = (int)(th % heads);
        const int t = (int)(th / heads);
        const int pos = start + t;
        if (pos < 0 || pos >= a.capacity) continue;
        if (hh < a.n_head + a.n_kv) {
            const bool is_q = hh < a.n_head;
            const int head = is_q ? hh : hh - a.n_head;
            const float *src = is_q ? a.q + ((size_t)t * a.n_head + head) * a.head_dim + 2 * pair
                                    : a.k + ((size_t)t * a.n_kv + head) * a.head_dim + 2 * pair;
            const float x0 = src[0];
            const float x1 = src[1];
            float y0 = x0, y1 = x1;
            if (2 * pair < a.n_rot) {
                const float angle = (float)pos * a.freq[pair];
                float s, c;
                sincosf(angle, &s, &c);
                y0 = x0 * c - x1 * s;
                y1 = x0 * s + x1 * c;
            }
            if (is_q) {
                float *dq = a.q + ((size_t)t * a.n_head + head) * a.head_dim + 2 * pair;
                dq[0] = y0;
                dq[1] = y1;
            } else {
                unsigned *dk = (unsigned *)(a.kcache + (size_t)pos * kv_dim + head * a.head_dim + 2 * pair);
                *dk = f16_bits(y0) | (f16_bits(y1) << 16);
            }
        } else {
            const int head = hh - a.n_head - a.n_kv;
            const float *src = a.v + (size_t)t * kv_dim + head * a.head_dim + 2 * pair;
            unsigned *dv = (unsigned *)(a.vcache + (size_t)pos * kv_dim + head * a.head_dim + 2 * pair);
            *dv = f16_bits(src[0]) | (f16_bits(src[1]) << 16);
        }
    }
}

// ---------------------------------------------------------------------------
// Decode attention for one token: workgroup (head, split) of W waves takes
// positions [begin, end) of the position + 1 visible ones, in chunks of
// 8 W NP rows (NP passes of 8 W rows).  Eight lanes share a row (16 bytes =
// 8 dims of it each), and a chunk's key AND value rows are all loaded before
// any arithmetic, so the whole chunk costs one memory latency:
//   scores: each lane's 8-dim partial dot (q in registers), summed over the
//           row's 8 lanes by xor shuffles (every lane of the row ends with the
//           same bits), then * scale (the reference's dot * scale);
//   softmax: the chunk's workgroup max m', the running state rescaled by
//           exp(m - m'), p = exp(s - m') -- with one chunk per split m is
//           -inf first, so p = exp(s - max) exactly as the reference forms it;
//   values: each lane accumulates p * v over its rows for its 8 dims; the row
//           slots are summed by xor shuffles in a wave and in LDS across waves,
//           in a fixed order, and so are the weights.
// Two shapes: 16 waves x 8 passes (1024-row chunks) for one split per head,
// 4 waves x 8 passes (256-row chunks) when the positions are split over
// workgroups, so a split of about 256 positions is one chunk (measured
// against 16 x 2 and 8 x 2 passes: equal at 600 positions, faster at 4096).
// splits == 1 writes acc / sum.  defer writes every split's unnormalised
// (acc, max, sum) for the next kernel to combine (the O projection's GEMV
// prologue).  Otherwise each workgroup stores them with agent-scope atomic
// stores and the last workgroup of the head to arrive (an arrival counter,
// reset by it) combines them:
//     max = max_s max_s;  e_s = exp(max_s - max);
//     out = (sum_s acc_s * e_s) / (sum_s sum_s * e_s)   (s ascending, fused
//     multiply-adds)
// -- the same arithmetic as one softmax summed in another order (gpu.cu
// attention_combine 735-762), and the same as the GEMV prologue's.
// ---------------------------------------------------------------------------
static __device__ __forceinline__ float wave_max(float v) {
    v = xor_max<32>(v);
    v = xor_max<16>(v);
    v = xor_max<8>(v);
    v = xor_max<4>(v);
    v = xor_max<2>(v);
    return xor_max<1>(v);
}
static __device__ __forceinline__ float wave_sum(float v) {
    v = xor_add<32>(v);
    v = xor_add<16>(v);
    v = xor_add<8>(v);
    v = xor_add<4>(v);
    v = xor_add<2>(v);
    return xor_add<1>(v);
}

// What the decode attention reads before its first key, as its leading
// kernel arguments: preloaded into SGPRs at wave launch (the kernarg preload
// the row-slice GEMVs use), so the cache position's load, the first dependent
// read, issues at once.  dims = n_head | n_kv << 16; cap = capacity | defer <<
// 31; the (max, sum) plane follows the partial sums (part_acc + heads * splits
// * 64).  scale, out and counters stay in the argument block.
struct AttnHead {
    const float *q;
    const uint16_t *kcache, *vcache;
    const int *position;
    float *part_acc;
    int dims, splits, cap;
};

template <int W, int NP>
static __device__ __forceinline__ void attn_decode_body(const AttnHead &hd, const Q8AttnDecodeArgs &a) {
    constexpr int T = 64 * W;
    constexpr int HD = Q8_ATTN_HEAD_DIM;
    constexpr int RP = T / 8;  // rows per pass
    __shared__ float red[W];
    __shared__ float lsum[W];
    __shared__ __attribute__((aligned(16))) float part[W][HD];
    __shared__ int last_flag;
    const int n_head_ = hd.dims & 0xffff;
    const int n_kv_ = hd.dims >> 16;
    const int splits_ = hd.splits;
    const int capacity_ = hd.cap & 0x7fffffff;
    const int defer_ = (int)((unsigned)hd.cap >> 31);
    float *const part_acc_ = hd.part_acc;
    float *const part_ms_ = hd.part_acc + (size_t)n_head_ * splits_ * Q8_ATTN_HEAD_DIM;
    const int position = *hd.position;
    // Workgroup -> (head, split).  The heads of a kv head read the same rows:
    // (kv head, split, head of the group), a contiguous run of them per XCD
    // (round-robin dispatch), leaves all but the first of a group their rows in
    // that XCD's L2: dealt over all eight, every XCD fetched the group's rows.
    // Four decode layers of 32 heads on 8: 129 -> 119 us at 3500 positions, 116
    // -> 110 at 1500; two heads a group or 300 positions: within 0.5%.  With a
    // kv head of its own a head shares nothing.
    const int gsize = n_head_ / n_kv_;
    int head = blockIdx.x / splits_;
    int split = blockIdx.x - head * splits_;
    int kvh = head;
    if (gsize > 1) {
        const int total = n_head_ * splits_;
        const int xcd = blockIdx.x & 7;
        const int item = xcd * (total >> 3) + min(xcd, total & 7) + (int)(blockIdx.x >> 3);
        const int pair = item / gsize;
        kvh = pair / splits_;
        split = pair - kvh * splits_;
        head = kvh * gsize + item - pair * gsize;
    }
    const int kv_dim = n_kv_ * HD;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int kc = tid & 7;     // dims 8 kc .. 8 kc + 7
    const int slot = tid >> 3;  // row slot of the pass
    const uint16_t *kbase = hd.kcache + kvh * HD + 8 * kc;
    const uint16_t *vbase = hd.vcache + kvh * HD + 8 * kc;
    float m = -INFINITY;  // running max, workgroup-uniform
    float l = 0.0f;       // this lane's weights summed over its rows
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    // One chunk: rows c0 + slot + RP j (j < NP), live below `end`.
    auto chunk = [&](int c0, int end, const f32x4 &q0, const f32x4 &q1, const i32x4 *ku, const i32x4 *vu) {
        float sc[NP];
        float cmax = -INFINITY;
#pragma unroll
        for (int j = 0; j < NP; j++) {
            float dot = 0.0f;
            dot = __builtin_fmaf(q0[0], f16_to_f32((unsigned)ku[j][0] & 0xffffu), dot);
            dot = __builtin_fmaf(q0[1], f16_to_f32((unsigned)ku[j][0] >> 16), dot);
            dot = __builtin_fmaf(q0[2], f16_to_f32((unsigned)ku[j][1] & 0xffffu), dot);
            dot = __builtin_fmaf(q0[3], f16_to_f32((unsigned)ku[j][1] >> 16), dot);
            dot = __builtin_fmaf(q1[0], f16_to_f32((unsigned)ku[j][2] & 0xffffu), dot);
            dot = __builtin_fmaf(q1[1], f16_to_f32((unsigned)ku[j][2] >> 16), dot);
            dot = __builtin_fmaf(q1[2], f16_to_f32((unsigned)ku[j][3] & 0xffffu), dot);
            dot = __builtin_fmaf(q1[3], f16_to_f32((unsigned)ku[j][3] >> 16), dot);
            dot = xor_add<1>(dot);
            dot = xor_add<2>(dot);
            dot = xor_add<4>(dot);
            sc[j] = dot * a.scale;
            if (c0 + slot + RP * j < end) cmax = fmaxf(cmax, sc[j]);
        }
        cmax = wave_max(cmax);
        if (lane == 0) red[wave] = cmax;
        __syncthreads();
        float mx = m;
#pragma unroll
        for (int w = 0; w < W; w++) mx = fmaxf(mx, red[w]);
        __syncthreads();  // red is rewritten by the next chunk
        const float f = expf(m - mx);  // 0 on the first chunk (m = -inf), when l and acc are 0
        l *= f;
#pragma unroll
        for (int d = 0; d < 8; d++) acc[d] *= f;
#pragma unroll
        for (int j = 0; j < NP; j++) {
            if (c0 + slot + RP * j < end) {
                const float pj = expf(sc[j] - mx);
                l += pj;
#pragma unroll
                for (int d = 0; d < 8; d++) {
                    const unsigned bits = ((unsigned)vu[j][d >> 1] >> (16 * (d & 1))) & 0xffffu;
                    acc[d] = __builtin_fmaf(pj, f16_to_f32(bits), acc[d]);
                }
            }
        }
        m = mx;
    };
    const int visible = min(position + 1, capacity_);
    const int per = (visible + splits_ - 1) / splits_;
    const int begin = split * per;
    const int end = min(begin + per, visible);
    // A chunk's key and value rows, clamped to the last live row: rows past
    // `end` repeat its address (no extra traffic) and are masked.  The first
    // chunk is issued before q is read, so a split of one chunk waits for one
    // memory latency; a later one once the previous is computed (its loads ahead
    // of that, in a second set of registers, gained nothing: four layers of 32
    // heads on 8 at 3500 positions 118.9 against 119.3 us, 36 on 36 146.5 both,
    // at 4000, on four waves, 160.7 against 157).
    i32x4 ku[NP], vu[NP];
    auto load_chunk = [&](int c0) {
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const int p = min(c0 + slot + RP * j, end - 1);
            ku[j] = *(const i32x4 *)(kbase + (size_t)p * kv_dim);
            vu[j] = *(const i32x4 *)(vbase + (size_t)p * kv_dim);
        }
    };
    if (begin < end) load_chunk(begin);
    const f32x4 q0 = *(const f32x4 *)(hd.q + (size_t)head * HD + 8 * kc);
    const f32x4 q1 = *(const f32x4 *)(hd.q + (size_t)head * HD + 8 * kc + 4);
    __builtin_amdgcn_sched_barrier(0);
    for (int c0 = begin; c0 < end; c0 += RP * NP) {
        chunk(c0, end, q0, q1, ku, vu);
        if (c0 + RP * NP < end) load_chunk(c0 + RP * NP);
    }
    // row slots of a wave (lanes with the same kc), then the waves; the
    // weights once per row (the kc == 0 lanes)
#pragma unroll
    for (int d = 0; d < 8; d++) {
        acc[d] = xor_add<8>(acc[d]);
        acc[d] = xor_add<16>(acc[d]);
        acc[d] = xor_add<32>(acc[d]);
    }
    const float lw = wave_sum(kc == 0 ? l : 0.0f);
    if (lane < 8) {
        *(f32x4 *)(&part[wave][8 * lane]) = (f32x4){acc[0], acc[1], acc[2], acc[3]};
        *(f32x4 *)(&part[wave][8 * lane + 4]) = (f32x4){acc[4], acc[5], acc[6], acc[7]};
    }
    if (lane == 0) lsum[wave] = lw;
    __syncthreads();
    if (wave != 0) {
        if (splits_ == 1 || defer_) return;
    }
    float tot = 0.0f, sum = 0.0f;
    if (wave == 0) {
#pragma unroll
        for (int w = 0; w < W; w++) tot += part[w][lane];
#pragma unroll
        for (int w = 0; w < W; w++) sum += lsum[w];
    }
    const float mx = m;
    const size_t base = (size_t)head * splits_;
    if (defer_) {  // wave 0: the next kernel reads these after this one ends
        part_acc_[(base + split) * HD + lane] = tot;
        if (lane == 0) {
            *(f32x2 *)(part_ms_ + 2 * (base + split)) = (f32x2){mx, sum};
        }
        return;
    }
    if (splits_ == 1) {
        a.out[(size_t)head * HD + lane] = tot / sum;
        return;
    }
    if (wave == 0) {
        store_agent(part_acc_ + (base + split) * HD + lane, tot);
        if (lane == 0) {
            store_agent(part_ms_ + 2 * (base + split), mx);
            store_agent(part_ms_ + 2 * (base + split) + 1, sum);
        }
    }
    // Release the partials at agent scope, count the arrival with an acq_rel
    // read-modify-write, and acquire in the last workgroup before its loads:
    // the XCDs' L2s are not coherent with each other, so the ordering has to
    // be stated, not left to the stores having completed.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    if (tid == 0) {
        const unsigned old = __hip_atomic_fetch_add(&a.counters[head], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        last_flag = (old == (unsigned)(splits_ - 1));
    }
    __syncthreads();
    if (!last_flag) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (tid == 0) __hip_atomic_store(&a.counters[head], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (wave != 0) return;
    float gmax = -INFINITY;
    for (int s = 0; s < splits_; s++) gmax = fmaxf(gmax, load_agent(part_ms_ + 2 * (base + s)));
    float num = 0.0f, den = 0.0f;
    for (int s = 0; s < splits_; s++) {
        const float f = expf(load_agent(part_ms_ + 2 * (base + s)) - gmax);  // an empty split has max -inf: f = 0
        den = __builtin_fmaf(load_agent(part_ms_ + 2 * (base + s) + 1), f, den);
        num = __builtin_fmaf(load_agent(part_acc_ + (base + s) * HD + lane), f, num);
    }
    a.out[(size_t)head * HD + lane] = num / den;
}

#define Q8_ATTN_PARAMS                                                                                     \
    const float *q, const uint16_t *kcache, const uint16_t *vcache, const int *position, float *part_acc, int dims, \
        int splits, int cap, Q8AttnDecodeArgs a
extern "C" __global__ __launch_bounds__(1024) void q8_attn_decode(Q8_ATTN_PARAMS) {
    attn_decode_body<16, 8>(AttnHead{q, kcache, vcache, position, part_acc, dims, splits, cap}, a);
}
extern "C" __global__ __launch_bounds__(256) void q8_attn_decode_w4(Q8_ATTN_PARAMS) {
    attn_decode_body<4, 8>(AttnHead{q, kcache, vcache, position, part_acc, dims, splits, cap}, a);
}
// The split kernel's 256-row chunks over eight waves: four rows a lane instead of eight.
extern "C" __global__ __launch_bounds__(512) void q8_attn_decode_w8(Q8_ATTN_PARAMS) {
    attn_decode_body<8, 4>(AttnHead{q, kcache, vcache, position, part_acc, dims, splits, cap}, a);
}

// ---------------------------------------------------------------------------
// Prefill attention: n query tokens at cache positions start .. start+n-1, each
// seeing keys 0 .. its own position (causal), on v_mfma_f32_32x32x16_f16.
//
// A workgroup is (head, 32 queries); its KS waves deal the 32-key tiles among
// themselves (wave g takes tiles g, g + KS, ...) and combine their (max, sum,
// output) through LDS at the end.  A wave's K and V tile go to its own 8 KB of
// LDS by direct loads (16 bytes a lane, whole 128-byte rows): the next K is
// loaded once the scores have read this one, the next V once the values have,
// so each has half a tile's time to arrive and no wave waits for another.
// Per tile a wave computes S^T = K Q^T (keys x queries) and O^T += V^T P^T
// (dims x queries), so a lane always holds one query (lane % 32): its scores,
// its running max and sum, and its output accumulators, and the softmax needs
// no transpose; the V^T operand is read transposed (ds_read_b64_tr_b16).  Rows
// of 128 bytes would put every row's 16-byte chunk c on the same banks, so row
// k keeps its chunk c at c ^ (k % 8).
//
// f32 operands enter the MFMA exactly as two f16 parts (x = hi + lo, hi =
// f16(x), lo = f16(x - hi), ~22 significant bits; products of f16 are exact
// in f32): q for the scores, the probabilities for the values; keys and
// values are the f16 cache itself.  Accumulation is f32.  Element k of an
// MFMA operand sits in lane-half k / 8, slot k % 8, for A and B alike; D[m][n]
// has n = lane % 32, m = 8(v/4) + 4(lane/32) + v%4.
//
// The softmax runs in base 2: q is multiplied by the fraction of scale log2(e)
// and the scores by a power of two (exact, so a row's maximum is the bits of one
// of its scores' products), and a weight is one fma and one v_exp_f32, with one
// rounding of the exponent's argument.  The query's own power of two goes the same
// way: its largest element is brought to 2^13 .. 2^14 before the split, where lo
// stays clear of the f16 subnormals for every element that counts.  Split at the
// query's own size the error was 2^-25 for elements below 1/4, and 1.4 times that
// behind the factor of scale 0.125: against 64 bits, queries of 0.01 on keys of 100
// 2.4e-6 (1.7e-6 without the factor, 2.2e-7 now), of 1 on 1 2.2e-7 as now.
// A row's reference m moves only when its tile max passes it by more than 8
// (weights stay below 2^8, sums in f32), so the accumulators are rescaled in few
// tiles; it starts finite, so that a row with no visible key yet subtracts no
// infinity.
// Heavier (later) query tiles of a head are launched first, and the workgroups
// of a head run on one XCD (round-robin dispatch), whose L2 then serves the
// head's cache rows to all of them.
//
// What bounds it: VALU and MFMA issue, about 1.55 us of a SIMD per 64 keys x
// 32 queries at four waves a SIMD (32 MFMAs 0.54 us, 33 v_exp_f32 and some 200
// other VALU the rest).  Against two waves a workgroup over 64-key tiles with
// V transposed in registers and a nine-instruction exp per weight, 36 heads:
// 512 tokens at 0 24.0 -> 13.8 us, 1000 at 3000 203 -> 96 us, 43 at 3000 72 ->
// 20 us.  64-key tiles (twice the LDS, three waves a SIMD at most): 14.3, 105
// and 20 us; two query tiles sharing a K/V tile in LDS: 15.0, 100 and 38 us.
// ---------------------------------------------------------------------------
#define Q8_ATTN_KEYS 32                                /* keys of a tile */
#define Q8_ATTN_TILE_BYTES (Q8_ATTN_KEYS * Q8_ATTN_HEAD_DIM * 2) /* of K, or of V */
#define Q8_ATTN_O_PITCH 33                             /* f32 per dim row of a wave's outputs in LDS */

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const uint8_t lds_bytes_t;
typedef __attribute__((address_space(3))) void attn_lds_t;

// c x as f16 hi + lo, two values an instruction where there is one; the remainder
// c x - hi by one mixed-precision fma, two values of hi a register, so that both
// parts are of the same hi.
static __device__ __forceinline__ void split_f16(const float *x, float c, f16x8 &hi, f16x8 &lo) {
    union Parts {
        unsigned w[4];
        f16x8 v;
    } hp, lp;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        hp.w[i] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){x[2 * i] * c, x[2 * i + 1] * c}, f16x2));
        float l0, l1;
        asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(l0) : "v"(x[2 * i]), "v"(c), "v"(hp.w[i]));
        asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
            : "=v"(l1)
            : "v"(x[2 * i + 1]), "v"(c), "v"(hp.w[i]));
        lp.w[i] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){l0, l1}, f16x2));
    }
    hi = hp.v;
    lo = lp.v;
}
// The same of x itself.
static __device__ __forceinline__ void split_f16(const float *x, f16x8 &hi, f16x8 &lo) {
    union Parts {
        unsigned w[4];
        f16x8 v;
    } hp, lp;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        hp.w[i] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){x[2 * i], x[2 * i + 1]}, f16x2));
        float l0, l1;
        asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(l0) : "v"(hp.w[i]), "v"(x[2 * i]));
        asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
            : "=v"(l1)
            : "v"(hp.w[i]), "v"(x[2 * i + 1]));
        lp.w[i] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){l0, l1}, f16x2));
    }
    hi = hp.v;
    lo = lp.v;
}

// The V^T operands of a 16-key step, dims 0-31 (v0) and 32-63 (v1): four
// transposed reads of 4 keys x 16 dims each, in one block with their wait (as
// builtins the compiler drains every direct load in flight before them, the
// next tile's too).  OFF: the step's byte offset in the tile.
template <int OFF>
static __device__ __forceinline__ void read_vt(unsigned a0, unsigned a1, f16x8 &v0, f16x8 &v1) {
    s16x4 p0, p1, p2, p3;
    asm volatile(
        "ds_read_b64_tr_b16 %0, %4 offset:%6\n\t"
        "ds_read_b64_tr_b16 %1, %4 offset:%7\n\t"
        "ds_read_b64_tr_b16 %2, %5 offset:%6\n\t"
        "ds_read_b64_tr_b16 %3, %5 offset:%7\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(p0), "=&v"(p1), "=&v"(p2), "=&v"(p3)
        : "v"(a0), "v"(a1), "i"(OFF), "i"(OFF + 8 * 128)
        : "memory");
    v0 = __builtin_bit_cast(f16x8, __builtin_shufflevector(p0, p1, 0, 1, 2, 3, 4, 5, 6, 7));
    v1 = __builtin_bit_cast(f16x8, __builtin_shufflevector(p2, p3, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int KS>
static __device__ __forceinline__ void attn_prefill_body(const Q8AttnPrefillArgs &a) {
    constexpr int HD = Q8_ATTN_HEAD_DIM;
    constexpr int COMB = HD * Q8_ATTN_O_PITCH * 4;  // a wave's outputs, over the tiles' LDS
    constexpr int PER_WAVE = COMB > 2 * Q8_ATTN_TILE_BYTES ? COMB : 2 * Q8_ATTN_TILE_BYTES;
    constexpr int LOADS = Q8_ATTN_KEYS / 8;  // direct loads of a tile
    __shared__ __attribute__((aligned(1024))) uint8_t smem[KS * PER_WAVE];
    __shared__ float xm[KS][32], xl[KS][32];
    const int lane = threadIdx.x & 63;
    const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5;
    const int r = lane & 31;
    // grid workgroup -> (head, query tile), a contiguous run of items per XCD
    const int total = a.n_head * a.qtiles;
    const int xcd = blockIdx.x & 7;
    const int item = xcd * (total >> 3) + min(xcd, total & 7) + (int)(blockIdx.x >> 3);
    const int head = item / a.qtiles;
    const int qt = a.qtiles - 1 - (item - head * a.qtiles);
    const int kvh = head / (a.n_head / a.n_kv);
    const int kv_dim = a.n_kv * HD;
    const int start = *a.position;
    const int qrow = qt * 32 + r;  // this lane's query
    const int qa = start + qrow;   // its cache position
    const bool qlive = qrow < a.n;

    const int kend = min(start + min(qt * 32 + 32, a.n), a.capacity);  // keys [0, kend)
    const int ntiles = (kend + Q8_ATTN_KEYS - 1) / Q8_ATTN_KEYS;
    const int groups = min(KS, ntiles);  // waves that hold a tile

    // Direct loads: load j of a tile brings rows 8j .. 8j+7, lane i row i / 8's
    // chunk (i % 8) ^ (i / 8).
    const int lrow = lane >> 3;
    const int lchunk = ((lane & 7) ^ lrow) * 8;
    const uint16_t *const khead = a.kcache + kvh * HD + lchunk;
    const uint16_t *const vhead = a.vcache + kvh * HD + lchunk;
    uint8_t *const kbuf = smem + kg * 2 * Q8_ATTN_TILE_BYTES;
    uint8_t *const vbuf = kbuf + Q8_ATTN_TILE_BYTES;
    auto load_tile = [&](const uint16_t *base, int t, uint8_t *dst) {
#pragma unroll
        for (int j = 0; j < LOADS; j++) {
            const int key = min(t * Q8_ATTN_KEYS + 8 * j + lrow, kend - 1);  // rows past the last repeat it (masked)
            __builtin_amdgcn_global_load_lds(base + (size_t)key * kv_dim, (attn_lds_t *)(dst + j * 1024), 16, 0, 0);
        }
    };
    // the wave's direct loads have landed: all of them, or all but the last tile half's
    auto landed = [&](bool all) {
        __builtin_amdgcn_sched_barrier(0);
        if (all)
            __builtin_amdgcn_s_waitcnt(Q8_VMCNT_IMM(0));
        else
            __builtin_amdgcn_s_waitcnt(Q8_VMCNT_IMM(LOADS));
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_sched_barrier(0);
    };
    // the wave's LDS reads have returned: the buffer may be loaded again
    auto reads_done = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_sched_barrier(0);
    };

    float m = -FLT_MAX, l = 0.0f;  // not above any finite score; l: this lane's half of the keys
    f32x16 o[2] = {};
    if (kg < groups) {
        // q's loads first (they need no position), then the first tile's
        f32x4 qv[8];
        {
            const float *src = a.q + ((size_t)min(qrow, a.n - 1) * a.n_head + head) * HD + 8 * h;
#pragma unroll
            for (int s = 0; s < 8; s++) qv[s] = *(const f32x4 *)(src + 16 * (s >> 1) + 4 * (s & 1));
        }
        __builtin_amdgcn_sched_barrier(0);
        load_tile(khead, kg, kbuf);
        load_tile(vhead, kg, vbuf);
        // Q^T operand, d-step s: q[qrow][16s + 8h .. +7] times q_mult and the row's
        // power of two, as f16 hi/lo; lo from the unrounded product (the last tile's
        // padding queries repeat the last one: their outputs are cleared at the end)
        float top_q = 0.0f;
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int i = 0; i < 4; i++) top_q = fmaxf(top_q, fabsf(qv[s][i]));
        top_q = xor_max<32>(top_q);
        const int qe = max(__builtin_amdgcn_frexp_expf(top_q), -100);  // 0 for 0; the power stays finite
        const float qm = __builtin_ldexpf(a.q_mult, 14 - qe);
        const float s2 = __builtin_ldexpf(1.0f, min(max(a.s_exp + qe - 14, -126), 127));
        f16x8 qhi[4], qlo[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            float x[8];
#pragma unroll
            for (int i = 0; i < 8; i++) x[i] = qv[2 * s + (i >> 2)][i & 3];
            split_f16(x, qm, qhi[s], qlo[s]);
        }
        const int lim = min(qa, kend - 1);  // last key this lane's query sees
        int koff[4];
#pragma unroll
        for (int s = 0; s < 4; s++) koff[s] = r * 128 + (((2 * s + h) ^ (r & 7)) << 4);
        // V^T: 16 lanes read 4 keys x 16 dims; lane i the 8 bytes of key i / 4, dims 4 (i % 4)
        unsigned voff[2];
        {
            const int i = lane & 15, key = 4 * h + (i >> 2);
#pragma unroll
            for (int dt = 0; dt < 2; dt++)
                voff[dt] = (unsigned)(uintptr_t)(lds_bytes_t *)vbuf + key * 128 +
                           (((4 * dt + 2 * ((lane >> 4) & 1) + ((i >> 1) & 1)) ^ key) << 4) + 8 * (i & 1);
        }
        f32x16 st;
        // O^T += V^T P^T over the 16 keys from 16 J
        auto values = [&](auto jc) {
            constexpr int J = decltype(jc)::value;
            // slots 0-3: keys 16J + 4h + ..; slots 4-7: keys 16J + 8 + 4h + ..
            float pv[8];
#pragma unroll
            for (int i = 0; i < 8; i++) pv[i] = st[8 * J + i];
            f16x8 phi, plo, v0, v1;
            split_f16(pv, phi, plo);
            read_vt<J * 16 * 128>(voff[0], voff[1], v0, v1);
            o[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v0, phi, o[0], 0, 0, 0);
            o[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v1, phi, o[1], 0, 0, 0);
            o[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v0, plo, o[0], 0, 0, 0);
            o[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v1, plo, o[1], 0, 0, 0);
        };
        for (int t = kg; t < ntiles; t += KS) {
            const bool next = t + KS < ntiles;
            landed(false);  // K (V may still be in flight)
            st = (f32x16){};
#pragma unroll
            for (int s = 0; s < 4; s++) {  // S^T: keys x queries
                const f16x8 kv = *(const f16x8 *)(kbuf + koff[s]);
                st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kv, qhi[s], st, 0, 0, 0);
                st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kv, qlo[s], st, 0, 0, 0);
            }
            reads_done();
            if (next) load_tile(khead, t + KS, kbuf);
            // a tile whose last key precedes the tile's first query needs no mask
            const int p0 = t * Q8_ATTN_KEYS;
            if (p0 + Q8_ATTN_KEYS - 1 > min(start + qt * 32, kend - 1)) {
#pragma unroll
                for (int v = 0; v < 16; v++) st[v] = p0 + 8 * (v >> 2) + 4 * h + (v & 3) <= lim ? st[v] : -INFINITY;
            }
            float top[2] = {st[0], st[1]};
#pragma unroll
            for (int v = 2; v < 16; v++) top[v & 1] = fmaxf(top[v & 1], st[v]);
            const float tm = xor_max<32>(fmaxf(top[0], top[1])) * s2;
            if (__ballot(tm > m + 8.0f)) {
                const float mn = fmaxf(m, tm);
                const float corr = __builtin_amdgcn_exp2f(m - mn);
                m = mn;
                l *= corr;
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    o[0][v] *= corr;
                    o[1][v] *= corr;
                }
            }
            float rs[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int v = 0; v < 16; v++) {
                st[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[v], s2, -m));
                rs[v & 3] += st[v];
            }
            l += (rs[0] + rs[1]) + (rs[2] + rs[3]);
            landed(!next);  // V (the next K may still be in flight)
            values(std::integral_constant<int, 0>{});
            values(std::integral_constant<int, 1>{});
            reads_done();
            if (next) load_tile(vhead, t + KS, vbuf);
        }
    }

    // Combine the waves' softmax states through LDS; the first two waves
    // finish one half of the dims each.
    float *const comb = reinterpret_cast<float *>(smem);
    __syncthreads();  // the tiles are read
    if (kg < groups) {
        const float lt = xor_add<32>(l);
        float *dst = comb + kg * HD * Q8_ATTN_O_PITCH;
#pragma unroll
        for (int dt = 0; dt < 2; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) dst[(32 * dt + 8 * (v >> 2) + 4 * h + (v & 3)) * Q8_ATTN_O_PITCH + r] = o[dt][v];
        if (h == 0) {
            xm[kg][r] = m;
            xl[kg][r] = lt;
        }
    }
    __syncthreads();
    static_assert(KS >= 2, "two waves finish the dims");
    if (kg > 1) return;
    const int dt = kg;
    float mt = xm[0][r];
    for (int k = 1; k < groups; k++) mt = fmaxf(mt, xm[k][r]);
    // res[4g + e]: dim 32 dt + 8 g + 4 h + e of this lane's query (0 for the
    // padding queries of the last tile)
    float res[16], lt = 0.0f;
#pragma unroll
    for (int v = 0; v < 16; v++) res[v] = 0.0f;
    for (int k = 0; k < groups; k++) {
        const float c = __builtin_amdgcn_exp2f(xm[k][r] - mt);
        lt = __builtin_fmaf(xl[k][r], c, lt);
        const float *src = comb + (k * HD + 32 * dt + 4 * h) * Q8_ATTN_O_PITCH + r;
#pragma unroll
        for (int v = 0; v < 16; v++) res[v] = __builtin_fmaf(src[(8 * (v >> 2) + (v & 3)) * Q8_ATTN_O_PITCH], c, res[v]);
    }
#pragma unroll
    for (int v = 0; v < 16; v++) res[v] = qlive ? res[v] / lt : 0.0f;
    if (a.out && qlive) {
        float *orow = a.out + ((size_t)qrow * a.n_head + head) * HD + 32 * dt + 4 * h;
#pragma unroll
        for (int g = 0; g < 4; g++)
            *(f32x4 *)(orow + 8 * g) = (f32x4){res[4 * g], res[4 * g + 1], res[4 * g + 2], res[4 * g + 3]};
    }
    if (a.xq) {
        // The head's 64 dims are Q8_0 blocks 2 head and 2 head + 1 of the
        // query's row, so this workgroup owns whole prepared units (32
        // queries x one block).  Unit half hh holds elements 8c + J[hh][q]
        // (J = {0,4,1,5}, {2,6,3,7}); this lane holds 8c + 4h + {0..3}, so
        // the pair (r, r + 32) trades two values per chunk, then quantizes
        // as q8_quantize does (quant_store, the block peak across the pair).
        const int nb = 2 * a.n_head;
        float e[4][4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float v0 = res[4 * c], v1 = res[4 * c + 1];
            const float v2 = res[4 * c + 2], v3 = res[4 * c + 3];
            const float p0 = __shfl_xor(v0, 32), p1 = __shfl_xor(v1, 32);
            const float p2 = __shfl_xor(v2, 32), p3 = __shfl_xor(v3, 32);
            e[0][c] = h == 0 ? v0 : p2;  // 8c + 0 | 8c + 2
            e[1][c] = h == 0 ? p0 : v2;  // 8c + 4 | 8c + 6
            e[2][c] = h == 0 ? v1 : p3;  // 8c + 1 | 8c + 3
            e[3][c] = h == 0 ? p1 : v3;  // 8c + 5 | 8c + 7
        }
        const float peak = xor_max<32>(half_peak(e));
        quant_store(e, peak, a.xq, a.xs, (size_t)qt * nb + 2 * head + dt, 32 * h + r, h == 0, a.f16);
    }
}

// Four waves a workgroup, or eight while every workgroup has a CU to itself
// (run_attn_prefill has the times).
extern "C" __global__ __launch_bounds__(256, 4) void q8_attn_prefill(Q8AttnPrefillArgs a) { attn_prefill_body<4>(a); }
extern "C" __global__ __launch_bounds__(512, 4) void q8_attn_prefill_k8(Q8AttnPrefillArgs a) {
    attn_prefill_body<8>(a);
}

// ---------------------------------------------------------------------------
// Synthetic Q8_0 blocks (GGUF byte layout) from a counter-based generator:
// SplitMix64 of (seed, block).  q = byte % 255 - 127 (uniform over
// [-127, 127] up to a 1/255 bias), d = f16(|z| * scale_std / 127) with z a
// Box-Muller normal.  Deterministic for a seed; not the host generator's
// stream (the oracle checks against the bytes read back from the device).
// ---------------------------------------------------------------------------
static __device__ __forceinline__ unsigned long long splitmix64(unsigned long long z) {
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

extern "C" __global__ __launch_bounds__(256) void q8_synth(Q8SynthArgs a) {
    for (long long b = (long long)blockIdx.x * blockDim.x + threadIdx.x; b < a.blocks;
         b += (long long)gridDim.x * blockDim.x) {
        uint8_t *dst = a.dst + b * Q8_BLOCK_BYTES;
        const unsigned long long h0 = splitmix64(a.seed ^ ((unsigned long long)b * 0xd1b54a32d192ed03ull));
        const float u1 = (float)((h0 >> 40) + 1) * (1.0f / 16777216.0f);  // (0, 1]
        const float u2 = (float)((h0 >> 16) & 0xffffffull) * (1.0f / 16777216.0f);
        const float z = sqrtf(-2.0f * logf(u1)) * cosf(6.28318530718f * u2);
        const unsigned d = f16_bits(fabsf(z) * a.scale_std / 127.0f);
        dst[0] = (uint8_t)(d & 0xff);
        dst[1] = (uint8_t)(d >> 8);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const unsigned long long h = splitmix64(h0 + (unsigned long long)(w + 1));
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int q = (int)((h >> (8 * e)) & 0xffull) % 255 - 127;
                dst[2 + 8 * w + e] = (uint8_t)(signed char)q;
            }
        }
    }
}

extern "C" __global__ __launch_bounds__(64) void q8_advance(Q8AdvanceArgs a) {
    if (threadIdx.x == 0) a.position[0] += a.advance;
}
