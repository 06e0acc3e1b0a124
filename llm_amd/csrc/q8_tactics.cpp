// q8_tactics.cpp -- see q8_tactics.h.
#include "q8_tactics.h"
#include "q8_layout.h"

#include <algorithm>
#include <cmath>

namespace {

const Q8TacticRow kRows[] = {
    {"matmul.gemv_f32", Q8_KERNEL_GEMV, 1, 1, Q8_MATURITY_MEASURED, 10,
     "n = 1 keeps f32 activations (tensor.rs:96-101); one 64-lane dwordx4 load per 32-row x "
     "32-element unit, x staged in LDS, HBM-bound"},
    {"matmul.gemm_mfma_i8", Q8_KERNEL_GEMM, 2, Q8_MAX_TOKENS, Q8_MATURITY_MEASURED, 10,
     "n >= 2 quantizes activations (tensor.rs:104-125); v_mfma_i32_32x32x32_i8 is one Q8_0 block "
     "per instruction, exact int32, scale products on v_mfma_f32_32x32x1_2b_f32"},
    {"matmul.gemv_q8x_two_tokens", Q8_KERNEL_GEMV, 2, 2, Q8_MATURITY_MEASURED, 9,
     "f32 x at n = 2 (q8_matmul without prepared activations; ranked below the GEMM, which plans for "
     "prepared activations keep): x quantized to Q8_0 in the GEMV's own launch, four v_dot4_i32_i8 per "
     "half block, the weight stream read once for both tokens; configs[1]'s W: 7.25 us against 10.45 us "
     "for quantize + int8 MFMA GEMM.  At n = 4 and 8 the quantization every workgroup repeats outgrew "
     "the GEMM (11.5 and 24.0 us against 10.5)"},
    {"matmul.gemm_mfma_f16", Q8_KERNEL_GEMM_F16, 2, Q8_MAX_TOKENS, Q8_MATURITY_EXPERIMENTAL, 5,
     "quants are integers |q| <= 127, exact in f16: two v_mfma_f32_32x32x16_f16 give each block's int32 "
     "dot already in f32, removing the 16 v_cvt_f32_i32 per 32x32 tile and block that bound the int8 "
     "path on the VALU; bit-identical to the int8 kernel.  Measured slower so far (gate|up n=512 70 us "
     "vs 50 us): one wave per row tile reads 2 KB of f16 activations per block-tile from LDS, about "
     "150 B/clk per CU at the MFMA rate, above the LDS bandwidth; option gemm.f16 = 1 selects it"},
    {"matmul.gemm_mfma_i8_pipelined", Q8_KERNEL_GEMM, 2, Q8_MAX_TOKENS, Q8_MATURITY_REJECTED, 0,
     "each item's MFMAs issued one item ahead of the previous epilogue (option gemm.pipe): two result "
     "buffers cost ~130 VGPRs, two waves per SIMD instead of three; gate|up n=512 57 us vs 51 us"},
    {"matmul.gemm_mfma_i8_lds_staged", Q8_KERNEL_GEMM, 2, Q8_MAX_TOKENS, Q8_MATURITY_REJECTED, 0,
     "int8 activations staged once per workgroup in LDS with global_load_lds and shared by row-tile "
     "waves (option gemm.lds), cutting L2 reads (the plain kernel reads both operands from L2 at "
     "86-92% hit rates, its HBM fetch 1.4-3.4x the weight bytes: the activations once per XCD): one "
     "workgroup barrier per block pair costs more; gate|up n=512 56 us vs 51 us"},
    {"matmul.gemm_f32_small_n", Q8_KERNEL_GEMM, 2, 7, Q8_MATURITY_REJECTED, 0,
     "the reference GPU's f32-activation path for 2 <= n <= 7 (cuda/mod.rs:883-891) disagrees with "
     "the CPU kernels that define parity, which quantize for every n >= 2"},
    {"matmul.gemm_mfma_i8_16x16x64", Q8_KERNEL_GEMM, 2, Q8_MAX_TOKENS, Q8_MATURITY_REJECTED, 0,
     "K = 64 sums two Q8_0 blocks with different d_w*d_x in one int32 accumulator, so the per-block "
     "scale can no longer be applied exactly"},
};
constexpr int kCount = sizeof(kRows) / sizeof(kRows[0]);

int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

int pairs_per_batch(int ppw) { return ppw <= 2 ? 2 : ppw <= 3 ? 3 : ppw <= 5 ? 5 : 3; }

}  // namespace

// GEMV launch shape: one workgroup per 32-row tile (two for the fused
// gate/up pair), its block pairs split over W waves.  Large matrices (two or
// more tiles per CU) take four waves of up to nine pairs; smaller ones take
// waves of about three pairs, up to 16 waves, so the whole matrix is in
// flight at once.  Splitting a tile's blocks over several workgroups (kslices)
// needs an agent-scope release per workgroup, which on gfx950 writes back the
// XCD's L2; measured slower, so it is never chosen here (option "gemv.slices").
void q8_gemv_shape(int out, int k, int cu_count, int slots, q8_tactic *t) {
    const int nb = k / 32;
    const int tiles = ceil_div(out, 32);
    const int npairs = ceil_div(nb, 2);
    const int cus = std::max(cu_count, 1);
    const int max_w = 16 / slots;
    // about three block pairs per wave, at any tile count: the lm_head
    // (122880 x 2304, 3840 tiles) measured 46.3 us at four waves per tile and
    // 42.7 us at twelve (one 301 MB copy, gfx950)
    int w = std::min(max_w, std::max(1, ceil_div(npairs, 3)));
    int ppw = ceil_div(npairs, w);
    if (ppw > 12) ppw = 12;  // LDS staging bound of a wave
    w = ceil_div(npairs, ppw);
    int s = 1;
    if (w > max_w) {  // K too long for one workgroup: split it
        s = ceil_div(w, max_w);
        const int pps = ceil_div(npairs, s);
        s = ceil_div(npairs, pps);
        w = ceil_div(pps, ppw);
    }
    t->kslices = s;
    t->waves_per_tile = w;
    t->pairs_per_wave = ppw;
    t->pairs_per_batch = pairs_per_batch(ppw);
    if (w * slots > 8 && t->pairs_per_batch == 9) t->pairs_per_batch = 5;
    // Blocks are summed in a fixed tree (deterministic, within f32 rounding of
    // the reference's left-to-right sum; every block value is the reference's
    // own bits).  exact = 1 (option "gemv.exact") keeps the reference's
    // left-to-right order for bit-identical outputs; it costs a serial chain of
    // nb adds per row at the end of the kernel (configs[0]: 5.48 vs 5.26 us).
    t->exact = 0;
    // A single matrix with fewer tiles than CUs runs in row slices (whole K
    // per workgroup): 8-row slices (four per tile) when 16-row slices would
    // already fill every CU and the 8-row workgroups fit (below), else
    // 16-row slices with as many waves as fit 16 at three loads per lane,
    // else six.  Measured
    // MALL-cold on gfx950 (tile kernel -> slices): configs[0] 5760 x 2304
    // 5.50 -> 5.36 us (16-row slices 5.50), O 2304 x 2304 4.98 -> 3.95 us
    // (8-row 4.29), down 2304 x 5760 8.25 -> 6.2 us (8-row 6.84); the lm_head
    // (3840 tiles) keeps the tile kernel (51.5 us either way).
    t->row_slice = Q8_TILE_ROWS;
    t->slice_loads = 0;
    // 8-row slices take two loads per lane (eight blocks a wave, more and
    // shorter waves) and only where every workgroup is resident at once, 32
    // waves a CU (eight per SIMD): configs[0] 5.13 -> 4.94 us against three
    // loads, 4096 x 2304 4.43 -> 4.22 us.  Where they would need a second
    // round of workgroups the 16-row slices win (6912 x 2304 with
    // non-temporal weight loads: 16-row 5.22 us, 8-row 5.37 at two loads and
    // 5.54 at three).
    const int w2 = ceil_div(nb, 2 * 4);
    if (slots == 1 && tiles < cus && 2 * tiles >= cus && w2 <= 16 && 4 * tiles <= cus * (32 / w2)) {
        t->row_slice = 8;
        t->slice_loads = 2;
    } else if (slots == 1 && tiles < cus) {
        if (ceil_div(nb, 3 * 2) <= 16) {
            t->row_slice = 16;
            t->slice_loads = 3;
        } else if (ceil_div(nb, 6 * 2) <= 16) {
            t->row_slice = 16;
            t->slice_loads = 6;
        }
    }
}

// GEMM launch shape.  A wave owns TPW token tiles of one 32-row tile and one
// of kwaves equal ranges of the block pairs; a workgroup holds the kwaves of one
// such tile, or of two neighbouring ones (twaves).
//
// What bounds it: a wave's pair takes 0.25 us (one token tile) or 0.45 us
// (two) alone and the launch about 7 us beside its pairs, so a small launch
// wants its pairs spread over waves, down to two each; a SIMD does one token
// tile's block in 76 ns from registers but 127 ns from the caches, two tiles'
// in 97 and 100, so a large one wants the two tiles that share the weight
// loads.  Between them the best launch has its waves resident at once (2800 of
// the 4096 at one token tile, 3072 at two): beyond, a second round of short
// waves pays the 7 us again.  kwaves is a power of two because other counts load
// the four SIMDs unevenly, and eight only while every workgroup has a CU to
// itself: a second one of eight waves doubles that CU's time (4608 x 2304 n = 64
// 9.4 us with eight, 8.6 with four).  From four to five workgroups a CU two waves
// each leave a SIMD with one more than the others, so rows of 32 pairs and more
// split over four there (3072 x 2304 n = 384 14.8 -> 13.9).  With two or four token
// tiles and one to two workgroups a CU, two neighbouring tiles share a workgroup
// and its weight loads in L1 (5760 x 2304 n = 64 9.4 -> 9.0, 4096 x 4096 n = 100 12.8 ->
// 12.0); where it leaves CUs idle it is 10 to 40% slower, and with more token
// tiles slower beside the riders of a layer (2304 x 5760 n = 192 by 1.8).  Four
// tiles per wave (two waves per SIMD) was never better.
//
// The lines are fit to gfx950 times over rows 200 .. 12000, K 512 .. 8192 and n
// 2 .. 1024, every shape of launch: 1120 calls with cold weights, 1.9% slower than
// the best on the geometric mean, and each projection of 119 decoder layers with
// their riders, 4.4%.  Eight waves up to 350 tiles, no paired tiles and two token
// tiles a wave from 1300 tiles and 80 000 tile-pairs gave 2.5% and 5.3%; about 18
// waves per CU with at least nine pairs a wave 14%.  Times of the three (the last
// first), us: 1152 x 896 n = 257 7.2, 5.7, 5.7; 5760 x 2304 n = 64 9.0, 9.4, 9.0;
// 2304 x 5760 n = 131 15.5, 13.4, 13.4; n = 1000 52.7, 47.6, 47.6.
void q8_gemm_shape(int n, int out, int k, int cu_count, q8_tactic *t) {
    const int nb = k / 32;
    const int npairs = ceil_div(nb, 2);
    const int ttiles = ceil_div(n, 32);
    const long long rtiles = ceil_div(out, 32);
    const long long cus = std::max(cu_count, 1);
    const long long tiles = rtiles * ttiles;
    // the lines lie at 870 tiles and 64 000 tile-pairs on 256 CUs
    const int tpw = (ttiles >= 2 && tiles * 256 >= 870 * cus && tiles * npairs * 256 >= 64000 * cus) ? 2 : 1;
    const long long groups = ceil_div(ttiles, tpw);
    const long long base = rtiles * groups;  // waves without a K split
    const long long most = (tpw == 1 ? 2800 : 3072) * cus / 256;
    const bool four = tpw == 1 && npairs >= 32 && base > 4 * cus && base <= 5 * cus;
    int kw = npairs < 8 ? 1 : tpw == 1 && base <= cus ? 8 : 4;  // rows below eight pairs were not measured and stay unsplit
    while (kw > 1 && ((base * kw > most && !(four && kw == 4)) || npairs < 2 * kw)) kw /= 2;
    const int ppw = ceil_div(npairs, kw);
    kw = ceil_div(npairs, ppw);
    t->tpw = tpw;
    t->twaves = (groups == 2 || groups == 4) && kw >= 2 && kw <= 4 && base > cus && base <= 2 * cus ? 2 : 1;
    t->kwaves = kw;
    t->kslices = 1;
    t->pairs_per_wave = ppw;
    t->smode = 1;
    t->xcd_remap = 1;
}

// A q, k, v group with its rotation in the epilogue: the plain group's K split
// (the results are its bits), one token tile a wave.  The epilogue is long and a
// wave of two token tiles runs it twice in a row (6912 x 2304 in a layer: n = 576
// 9 us more, n = 1000 7 more); only on long rows past twenty tiles a CU are the
// shared weight loads worth as much (12288 x 4096 n = 507 88.9 -> 75.7, n = 1000 172 ->
// 146; in a layer 1 and 16 us less).  From 128 row tiles up two token-tile waves
// share a workgroup and its weight loads where the token tiles pair off (in a
// layer at n = 43 0.6 us less; 3 us more where one wave idles, n = 257), up to the
// workgroup's 16 waves (the rule splits K over eight at most, an option over more).
void q8_gemm_rope_shape(int n, int out, int k, int cu_count, q8_tactic *t) {
    const int rtiles = ceil_div(out, 32), ttiles = ceil_div(n, 32);
    if (t->tpw == 2 && k >= 40 * 64 && (long long)rtiles * ttiles > 20LL * std::max(cu_count, 1)) return;
    t->tpw = 1;
    t->twaves = (rtiles >= 128 && ttiles % 2 == 0 && t->kwaves <= 8) ? 2 : 1;
}

// The fused gate/up launch (one wave a gate tile, its up tile and one token
// tile).  Four K waves while 2500 of them are enough for it, two up to six tiles
// a CU (fewer pairs and a reduction beat a wave of the whole row: 2304 x 1536 n = 550
// 20.9 -> 18.6 us).  Long rows (80 pairs) take four up to five tiles a CU (4096 x 5760
// n = 191 37.4 -> 32.4) and eight up to half a tile (256 x 5120 n = 257 13.6 -> 12.1);
// eight were slower elsewhere.  Over widths 256 .. 8192, K 512 .. 8192 and n 2 .. 1024
// (460 shapes) within 1.3% of the best on the geometric mean; four and two waves up
// to 2.4 and 4.9 tiles alone 2.2%, 11 waves per CU with nine pairs a wave 13%.
int q8_gemm_silu_kwaves(int n, int ffn, int k, int cu_count) {
    const int npairs = ceil_div(k / 32, 2);
    const long long base = (long long)ceil_div(ffn, 32) * ceil_div(n, 32);
    const long long cus = std::max(cu_count, 1);
    const bool lng = npairs >= 80;
    int kw = npairs < 8 ? 1 : lng && 2 * base <= cus ? 8 : 4;
    if (kw == 4 && (lng ? base > 5 * cus : base * 4 * 256 > 2500 * cus)) kw = 2;
    if (kw == 2 && base > 6 * cus) kw = 1;
    while (kw > 1 && npairs < 2 * kw) kw /= 2;
    return kw;
}

// f16 GEMM launch shape: TPW token tiles per wave (2 when there are two or
// more), RW row-tile waves sharing the LDS-staged activations, KW K-split
// waves, RW * KW <= 8.  The GEMM kernel runs two waves per SIMD (about 210
// VGPRs), so the chip holds 2 * 4 * cu_count waves at once; the search takes
// the (RW, KW) whose last round of waves is fullest, discounted for the fixed
// per-wave cost (about two block pairs of prologue, drain and K reduction).
void q8_gemm_h_shape(int n, int out, int k, int cu_count, q8_tactic *t) {
    q8_gemm_staged_shape(n, out, k, cu_count, 0, t);
}

void q8_gemm_staged_shape(int n, int out, int k, int cu_count, int i8, q8_tactic *t) {
    const int nb = k / 32;
    const int npairs = ceil_div(nb, 2);
    const int ttiles = ceil_div(n, 32);
    const int rtiles = ceil_div(out, 32);
    const double cap = 2.0 * 4.0 * std::max(cu_count, 1);
    const int tpw = ttiles >= 2 ? 2 : 1;
    double best = -1.0;
    int best_rw = (tpw == 1 && i8) ? 2 : 4, best_kw = 1;
    for (int rw : {2, 4}) {
        if (tpw == 1 && rw != (i8 ? 2 : 4)) continue;  // built: f16 t1_r4, t2_r2, t2_r4; int8 t1_r2, t2_r2, t2_r4
        for (int kw = 1; rw * kw <= 8 && kw <= npairs; kw++) {
            // LDS: KW K groups x the staging ring, within 64 KB
            const long long lds =
                (long long)kw * Q8_GEMM_H_STAGES * (i8 ? Q8_GEMM_L_BUF_BYTES(tpw, rw) : Q8_GEMM_H_BUF_BYTES(tpw, rw));
            if (lds > 65536) continue;
            const int ppw = ceil_div(npairs, kw);
            if (ceil_div(npairs, ppw) != kw) continue;  // no K wave without pairs
            const double waves = (double)ceil_div(rtiles, rw) * ceil_div(ttiles, tpw) * rw * kw;
            const double rounds = waves / cap;
            const double fill = rounds / std::ceil(rounds);
            const double live = (double)rtiles / (ceil_div(rtiles, rw) * rw);  // row waves past the end idle
            const double score = fill * live * ppw / (ppw + 2.0);
            if (score > best + 1e-9) {
                best = score;
                best_rw = rw;
                best_kw = kw;
            }
        }
    }
    t->tpw = tpw;
    t->rwaves = best_rw;
    t->kwaves = best_kw;
    t->pairs_per_wave = ceil_div(npairs, best_kw);
    t->twaves = 1;
    t->kslices = 1;
    t->smode = 1;
    t->xcd_remap = 1;
}

int q8_tactics_for_kernel(int kernel, int n, int out, int k, int cu_count, q8_tactic *t) {
    for (int i = 0; i < kCount; i++) {
        const Q8TacticRow &row = kRows[i];
        if (row.kernel != kernel || row.maturity == Q8_MATURITY_REJECTED) continue;
        *t = q8_tactic{};
        t->kernel = kernel;
        t->name = row.name;
        t->evidence = row.evidence;
        if (kernel == Q8_KERNEL_GEMV)
            q8_gemv_shape(out, k, cu_count, 1, t);
        else if (kernel == Q8_KERNEL_GEMM_F16)
            q8_gemm_h_shape(n, out, k, cu_count, t);
        else
            q8_gemm_shape(n, out, k, cu_count, t);
        return Q8_OK;
    }
    return Q8_ERR_UNSUPPORTED;
}

int q8_tactics_prepared_format(int n) {
    q8_tactic t{};
    if (q8_tactics_choose(n, 32, 32, 1, &t) != Q8_OK) return Q8_PREPARED_I8;
    return t.kernel == Q8_KERNEL_GEMM_F16 ? Q8_PREPARED_F16 : Q8_PREPARED_I8;
}

int q8_tactics_table_size() { return kCount; }

const Q8TacticRow &q8_tactics_row(int i) { return kRows[i]; }

int q8_tactics_choose(int n, int out, int k, int cu_count, q8_tactic *t) {
    const Q8TacticRow *best = nullptr;
    for (int i = 0; i < kCount; i++) {
        const Q8TacticRow &row = kRows[i];
        if (row.maturity == Q8_MATURITY_REJECTED) continue;
        if (n < row.n_min || n > row.n_max) continue;
        if (!best || row.rank > best->rank) best = &row;
    }
    if (!best) return Q8_ERR_UNSUPPORTED;
    *t = q8_tactic{};
    t->kernel = best->kernel;
    t->name = best->name;
    t->evidence = best->evidence;
    if (best->kernel == Q8_KERNEL_GEMV)
        q8_gemv_shape(out, k, cu_count, 1, t);
    else if (best->kernel == Q8_KERNEL_GEMM_F16)
        q8_gemm_h_shape(n, out, k, cu_count, t);
    else
        q8_gemm_shape(n, out, k, cu_count, t);
    return Q8_OK;
}
