// Log-mel front end on the device: 16 kHz samples -> the [n_mel, n_len] input of the encoder's conv stem
// (log_mel_spectrogram, src/whisper.cpp:3181-3270, and its worker :3113-3179).
//
// The reference extends the signal by 200 reflected samples in front and 30 s + 200 samples of zeros behind, takes
// 400-sample frames every 160 samples under a periodic Hann window, a 400-point transform per frame (f32, halved down
// to 25-point sums), the power of bins 0 .. 200, a [n_mel, 201] filter bank, log10(max(., 1e-10)), and finally raises
// everything below (global maximum - 8) to it and maps x to (x + 4) / 4.
//
// Here everything up to the stored f32 is f64, where the reference's f32 transform is within about 1e-6 of the exact value.
// Two launches: k_log_mel_frames writes (log10 + 4) / 4 of every value and each workgroup's maximum, k_log_mel_finish raises
// what lies below the floor (the map is monotonic, so the floor is mapped and compared) and fills the frames past the end of
// the signal, which are log10(1e-10) by definition.
//
// k_log_mel_frames: 20 lanes take a pair of frames as the real and the imaginary part of one 400-point transform, 400 =
// 20 x 20: lane t transforms samples t + 20 j in registers, twiddles, the 20 x 20 values change lanes through LDS, lane c
// transforms again and holds bins c + 20 l.  A 20-point transform is 5 four-point and 4 five-point ones without twiddles
// between them (4 and 5 are coprime: Good's mapping).  The pair's spectra come apart through bin 400 - k, which lane 20 - c
// holds: ten values per lane through LDS.  The three pairs of a wavefront need no barrier.  Then a thread per (frame, band)
// sums the band's range of nonzero filter weights over the powers in LDS.
// What bounds it: f64 issue and, between the steps of a round, LDS and load latency, so three workgroups share a CU (168 registers,
// 52 KB of LDS), a sample that both frames of a pair want is loaded once, and the filter weights that are not zero lie in LDS
// (read from memory one by one they were a third of the time).  An hour of audio, 80 bands, both launches: 376 us (600 with the
// weights in memory and two workgroups to a CU; by direct sums, 0.32 M multiply-adds a frame instead of 8 k operations, 4.2 ms);
// 128 bands 520; 3 s 18 us, nearly all of it the latency of one round and of the launches.
#include "common.h"

#define MEL_NFFT   400
#define MEL_HOP    160
#define MEL_BINS   201
#define MEL_PAIRS  12           // pairs of frames per workgroup and round: three in each of four wavefronts
#define MEL_FRAMES (2 * MEL_PAIRS)
#define MEL_LD     21           // values between the rows of a pair's 20 x 20 exchange (20 would put a column on 8 banks)
#define MEL_PAIR_LD (20 * MEL_LD)                       // holds the exchange, later the powers of both frames (2 x 201)
#define MEL_MAX_BANDS 128
#define MEL_GROUPS 768          // workgroups at most: three to a CU; each walks a run of consecutive rounds
#define MEL_LOG_BITS 6
#define MEL_WEIGHTS 224         // nonzero filter weights in LDS for a wavefront's share of the bands (a bin belongs to two of the usual triangles: about 100)

typedef double double2_t __attribute__((ext_vector_type(2)));

struct cplx { double re, im; };
__device__ __forceinline__ cplx cadd(cplx a, cplx b) { return { a.re + b.re, a.im + b.im }; }
__device__ __forceinline__ cplx csub(cplx a, cplx b) { return { a.re - b.re, a.im - b.im }; }
__device__ __forceinline__ cplx cmul(cplx a, double2_t w) { return { __builtin_fma(a.re, w.x, -(a.im * w.y)), __builtin_fma(a.re, w.y, a.im * w.x) }; }

// X[k] = sum x[n] exp(-2 pi i n k / 4), in place
__device__ __forceinline__ void dft4(cplx & a, cplx & b, cplx & c, cplx & d) {
    const cplx s = cadd(a, c), t = csub(a, c), u = cadd(b, d), v = csub(b, d);
    a = cadd(s, u); c = csub(s, u);
    b = { t.re + v.im, t.im - v.re }; d = { t.re - v.im, t.im + v.re };
}
__device__ __forceinline__ void dft5(cplx & x0, cplx & x1, cplx & x2, cplx & x3, cplx & x4) {
    constexpr double C1 = 0.30901699437494742410, C2 = -0.80901699437494742410, S1 = 0.95105651629515357212, S2 = 0.58778525229247312917;
    const cplx a = cadd(x1, x4), b = cadd(x2, x3), c = csub(x1, x4), d = csub(x2, x3);
    const cplx p = { __builtin_fma(C2, b.re, __builtin_fma(C1, a.re, x0.re)), __builtin_fma(C2, b.im, __builtin_fma(C1, a.im, x0.im)) };
    const cplx q = { __builtin_fma(C1, b.re, __builtin_fma(C2, a.re, x0.re)), __builtin_fma(C1, b.im, __builtin_fma(C2, a.im, x0.im)) };
    const cplx r = { __builtin_fma(S2, d.re, S1 * c.re), __builtin_fma(S2, d.im, S1 * c.im) };
    const cplx s = { __builtin_fma(-S1, d.re, S2 * c.re), __builtin_fma(-S1, d.im, S2 * c.im) };
    x0 = cadd(x0, cadd(a, b));
    x1 = { p.re + r.im, p.im - r.re }; x4 = { p.re - r.im, p.im + r.re };
    x2 = { q.re + s.im, q.im - s.re }; x3 = { q.re - s.im, q.im + s.re };
}
// X[k] = sum x[n] exp(-2 pi i n k / 20): n = 5 a + 4 b (mod 20), k = k mod 4 and k mod 5
__device__ __forceinline__ void dft20(cplx (&x)[20]) {
    cplx y[4][5];
#pragma unroll
    for (int b = 0; b < 5; ++b) {
#pragma unroll
        for (int a = 0; a < 4; ++a) y[a][b] = x[(5 * a + 4 * b) % 20];
        dft4(y[0][b], y[1][b], y[2][b], y[3][b]);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        dft5(y[a][0], y[a][1], y[a][2], y[a][3], y[a][4]);
#pragma unroll
        for (int b = 0; b < 5; ++b) x[(5 * a + 16 * b) % 20] = y[a][b];      // the k with k mod 4 = a and k mod 5 = b
    }
}

// log10(x) for x >= 1e-10 by table (P. T. P. Tang, ACM TOMS 16:4, 1990): x = 2^e m, c the middle of m's 1/64 of [1, 2),
// log10 m = log10 c + log1p(m / c - 1) / ln 10, |m / c - 1| < 2^-7.  `tab`: (1 / c, -log10(1 / c)).  Within 1e-15.
__device__ __forceinline__ double mel_log10(double x, const double2_t * __restrict__ tab) {
    const uint64_t bits = (uint64_t) __double_as_longlong(x);
    const int e = (int)(bits >> 52) - 1023;
    const double m = __longlong_as_double((long long)((bits & 0x000fffffffffffffull) | 0x3ff0000000000000ull));
    const double2_t t = tab[(bits >> (52 - MEL_LOG_BITS)) & ((1 << MEL_LOG_BITS) - 1)];
    const double r = __builtin_fma(m, t.x, -1.0);
    double p = __builtin_fma(r, 1.0 / 7, -1.0 / 6);
    p = __builtin_fma(p, r, 1.0 / 5); p = __builtin_fma(p, r, -1.0 / 4); p = __builtin_fma(p, r, 1.0 / 3); p = __builtin_fma(p, r, -1.0 / 2);
    p = __builtin_fma(p * r, r, r);
    const double y = __builtin_fma(p, 0.43429448190325182765, __builtin_fma((double) e, 0.30102999566398119521, t.y));
    return e < 1024 ? y : x;                            // infinity stays infinity
}

// the values of one lane visible to the other lanes of its wavefront (LDS accesses of a wavefront are carried out in order)
__device__ __forceinline__ void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); }

__global__ void __launch_bounds__(256, 3) k_log_mel_frames(const float * __restrict__ samples, int64_t n_samples, const float * __restrict__ filters,
                                                       int n_mel, int64_t n_frames, int64_t n_len, int64_t rounds_per_group,
                                                       float * __restrict__ mel, float * __restrict__ maxima) {
    __shared__ __attribute__((aligned(16))) double    xch[MEL_PAIRS * MEL_PAIR_LD];
    __shared__ __attribute__((aligned(16))) double2_t cs[MEL_NFFT];                // (cos, -sin)(2 pi i / 400)
    __shared__ __attribute__((aligned(16))) double2_t lt[1 << MEL_LOG_BITS];
    __shared__ int16_t range[MEL_MAX_BANDS][3];                                    // a band's nonzero weights: first, one past the last, place in weights (or -1)
    __shared__ float weights[4 * MEL_WEIGHTS];
    __shared__ float wmax[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    for (int i = tid; i < MEL_NFFT; i += 256) {
        double s, c;
        sincospi(2.0 * i / MEL_NFFT, &s, &c);
        cs[i] = (double2_t){ c, -s };
    }
    if (tid < 1 << MEL_LOG_BITS) {
        const double inv = 1.0 / (1.0 + (tid + 0.5) / (1 << MEL_LOG_BITS));
        lt[tid] = (double2_t){ inv, -log10(inv) };
    }
    // Mel filters are triangles over a few bins, and a zero weight adds nothing: each wavefront looks through every fourth band,
    // eight bands' rows requested at a time, and puts the nonzero ranges side by side in LDS (one that does not fit stays in memory;
    // all of them for a single round: 3 s of audio 18.1 us, 18.8 with the weights moved first).
    int used = 0;                                       // of this wavefront's share of weights
    for (int j0 = wave; j0 < n_mel; j0 += 32) {
        float w[8][4];
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const int j = j0 + 4 * b < n_mel ? j0 + 4 * b : n_mel - 1;
#pragma unroll
            for (int i = 0; i < 4; ++i) { const int k = lane + 64 * i; w[b][i] = filters[j * MEL_BINS + (k < MEL_BINS ? k : MEL_BINS - 1)]; }
        }
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            int first = MEL_BINS, last = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint64_t any = __ballot(w[b][i] != 0.0f && lane + 64 * i < MEL_BINS);
                if (any) { first = min(first, 64 * i + (int) __builtin_ctzll(any)); last = 64 * i + 64 - (int) __builtin_clzll(any); }
            }
            first = min(first, last);
            if (j0 + 4 * b >= n_mel) break;
            const int at = rounds_per_group > 1 && used + last - first <= MEL_WEIGHTS ? wave * MEL_WEIGHTS + used : -1;
            if (lane == 0) { range[j0 + 4 * b][0] = (int16_t) first; range[j0 + 4 * b][1] = (int16_t) last; range[j0 + 4 * b][2] = (int16_t) at; }
            if (at >= 0) {
                used += last - first;
#pragma unroll
                for (int i = 0; i < 4; ++i) { const int k = lane + 64 * i; if (k >= first && k < last) weights[at + k - first] = w[b][i]; }
            }
        }
    }
    __syncthreads();

    const int slot = lane < 60 ? lane / 20 : 2, t = lane < 60 ? lane % 20 : lane - 60;    // (lanes 60 .. 63 do what lanes 40 .. 43 do)
    const int pair = wave * 3 + slot;
    double * my = xch + pair * MEL_PAIR_LD;
    float vmax = -INFINITY;
    const int64_t round0 = (int64_t) blockIdx.x * rounds_per_group;
#pragma unroll 1
    for (int64_t round = round0; round < round0 + rounds_per_group; ++round) {
        const int64_t i0 = round * MEL_FRAMES;
        if (i0 >= n_frames) break;
        cplx z[20];
        {
            // sample n = t + 20 j of frames A = i0 + 2 pair and A + 1; position in the signal: reflected head, the samples, zeros
            const int64_t p0 = (i0 + 2 * pair) * MEL_HOP + t - MEL_NFFT / 2;
            float x[28];                                // (frame A + 1 begins at A's sample 160: j = 8)
            if (i0 * MEL_HOP >= MEL_NFFT / 2 && (i0 + MEL_FRAMES - 1) * MEL_HOP + MEL_NFFT / 2 <= n_samples) {
                const float * sp = samples + p0;
#pragma unroll
                for (int j = 0; j < 28; ++j) x[j] = sp[20 * j];
            } else {
                auto at = [&](int64_t p) __attribute__((always_inline)) {
                    int64_t i = p < 0 ? -p : p;
                    i = i < n_samples ? i : n_samples - 1;
                    const float x = samples[i];
                    return p < n_samples ? x : 0.0f;
                };
#pragma unroll
                for (int j = 0; j < 28; ++j) x[j] = at(p0 + 20 * j);
            }
#pragma unroll
            for (int j = 0; j < 20; ++j) {
                const double w = 0.5 * (1.0 - cs[t + 20 * j].x);
                z[j] = { w * (double) x[j], w * (double) x[j + 8] };
            }
        }
        // (no instruction moves across: twiddles read ahead of their step would cost the registers of a third workgroup on the CU)
        __builtin_amdgcn_sched_barrier(0);
        dft20(z);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 1; c < 20; ++c) z[c] = cmul(z[c], cs[t * c]);
        __builtin_amdgcn_sched_barrier(0);
        // 20 x 20 values change lanes, real parts first
#pragma unroll
        for (int c = 0; c < 20; ++c) my[c * MEL_LD + t] = z[c].re;
        wave_fence();
#pragma unroll
        for (int c = 0; c < 20; ++c) z[c].re = my[t * MEL_LD + c];
        wave_fence();
#pragma unroll
        for (int c = 0; c < 20; ++c) my[c * MEL_LD + t] = z[c].im;
        wave_fence();
#pragma unroll
        for (int c = 0; c < 20; ++c) z[c].im = my[t * MEL_LD + c];
        wave_fence();
        dft20(z);                                       // z[l]: bin t + 20 l
        // upper halves to the lane that holds the mirrored bins
#pragma unroll
        for (int l = 0; l < 10; ++l) { my[2 * l * 20 + t] = z[10 + l].re; my[(2 * l + 1) * 20 + t] = z[10 + l].im; }
        wave_fence();
        const int mirror = t == 0 ? 0 : 20 - t;
        double pa[10], pb[10], pa_last = 0.0, pb_last = 0.0;
        auto power = [](cplx a, cplx b, double & fa, double & fb) __attribute__((always_inline)) {   // b: bin 400 - k
            const double re0 = a.re + b.re, im0 = a.im - b.im, re1 = a.im + b.im, im1 = b.re - a.re;
            fa = 0.25 * __builtin_fma(re0, re0, im0 * im0); fb = 0.25 * __builtin_fma(re1, re1, im1 * im1);
        };
#pragma unroll
        for (int l = 0; l < 10; ++l) {
            // 400 - (t + 20 l) = mirror + 20 (19 - l), or, for t = 0, 20 (20 - l) (bin 0 is its own mirror)
            const int up = t == 0 ? 10 - l : 9 - l;     // index among the upper halves
            const int row = up < 10 ? up : 0;
            cplx b = { my[2 * row * 20 + mirror], my[(2 * row + 1) * 20 + mirror] };
            if (up == 10) b = z[0];
            power(z[l], b, pa[l], pb[l]);
        }
        if (t == 0) power(z[10], z[10], pa_last, pb_last);
        wave_fence();
#pragma unroll
        for (int l = 0; l < 10; ++l) { const int k = t + 20 * l; my[k] = pa[l]; my[MEL_BINS + k] = pb[l]; }
        if (t == 0) { my[200] = pa_last; my[MEL_BINS + 200] = pb_last; }
        __syncthreads();

        // filter bank: consecutive threads take consecutive frames of a band
        for (int p = tid; p < n_mel * MEL_FRAMES; p += 256) {
            const int j = p / MEL_FRAMES, f = p % MEL_FRAMES;
            const double * pw = xch + (f >> 1) * MEL_PAIR_LD + (f & 1) * MEL_BINS;
            const float * fl = filters + j * MEL_BINS;
            double sum = 0.0;
            const int first = range[j][0], last = range[j][1], at = range[j][2];
            auto add = [&](auto * fl) __attribute__((always_inline)) {         // fl[k]: the weight of bin k; four reads of each kind on their way
                int k = first;
                for (; k + 3 < last; k += 4) {
                    const double p0 = pw[k], p1 = pw[k + 1], p2 = pw[k + 2], p3 = pw[k + 3];
                    const float f0 = fl[k], f1 = fl[k + 1], f2 = fl[k + 2], f3 = fl[k + 3];
                    sum = __builtin_fma(p3, (double) f3, __builtin_fma(p2, (double) f2, __builtin_fma(p1, (double) f1, __builtin_fma(p0, (double) f0, sum))));
                }
                for (; k < last; ++k) sum = __builtin_fma(pw[k], (double) fl[k], sum);
            };
            if (at >= 0) add(weights + at - first); else add(filters + j * MEL_BINS);
            if (i0 + f < n_frames) {
                const float v = (float) mel_log10(sum > 1e-10 ? sum : 1e-10, lt);
                mel[(int64_t) j * n_len + i0 + f] = (float)(((double) v + 4.0) / 4.0);
                vmax = fmaxf(vmax, v);
            }
        }
        __syncthreads();                                // the powers are read before the next round's exchange
    }
    vmax = wave_max(vmax);
    if (lane == 0) wmax[wave] = vmax;
    __syncthreads();
    if (tid == 0) maxima[blockIdx.x] = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
}

// Values below (maximum - 8) are raised to it; frames past the signal hold log10(1e-10).  Reads every value and stores only
// those that change.  One band per blockIdx.y.
#define MEL_FINISH 8            // values per thread
__global__ void __launch_bounds__(256) k_log_mel_finish(float * __restrict__ mel, int64_t n_frames, int64_t n_len, const float * __restrict__ maxima, int n_maxima) {
    __shared__ float wmax[4];
    const int tid = threadIdx.x;
    const int64_t i0 = (int64_t) blockIdx.x * (256 * MEL_FINISH) + tid;
    float * row = mel + (int64_t) blockIdx.y * n_len;
    float y[MEL_FINISH];
#pragma unroll
    for (int r = 0; r < MEL_FINISH; ++r) { const int64_t i = i0 + 256 * r; y[r] = row[i < n_frames ? i : n_frames - 1]; }
    float top = -INFINITY;
    for (int g = tid; g < n_maxima; g += 256) top = fmaxf(top, maxima[g]);
    top = wave_max(top);
    if ((tid & 63) == 0) wmax[tid >> 6] = top;
    __syncthreads();
    top = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    if (n_frames < n_len) top = fmaxf(top, -10.0f);
    auto map = [](float x) __attribute__((always_inline)) { return (float)(((double) x + 4.0) / 4.0); };
    const float low = map((float)((double) top - 8.0)), past = fmaxf(map(-10.0f), low);
#pragma unroll
    for (int r = 0; r < MEL_FINISH; ++r) {
        const int64_t i = i0 + 256 * r;
        if (i < n_frames) { if (y[r] < low) row[i] = low; }
        else if (i < n_len) row[i] = past;
    }
}

extern "C" int64_t mi355x_log_mel_n_len(int64_t n_samples) { return n_samples > 0 ? (n_samples + 30 * 16000) / MEL_HOP : 0; }

extern "C" size_t mi355x_log_mel_workspace_size(int n_mel) {
    if (n_mel < 1 || n_mel > MEL_MAX_BANDS) return 0;
    return (size_t) MEL_GROUPS * sizeof(float);
}

extern "C" int mi355x_log_mel_spectrogram(const float * samples, int64_t n_samples, const float * filters, int n_mel, float * mel,
                                          void * workspace, size_t workspace_size, void * stream) {
    if (!samples || !filters || !mel) return MI355X_ERR_INVALID;
    if (n_mel < 1 || n_mel > MEL_MAX_BANDS) return MI355X_ERR_UNSUPPORTED;
    if (n_samples <= MEL_NFFT / 2 || n_samples > (int64_t) 1 << 40) return MI355X_ERR_INVALID;      // the reflected head reads samples 1 .. 200
    if (!workspace || workspace_size < mi355x_log_mel_workspace_size(n_mel) || (uintptr_t) workspace % 16 != 0) return MI355X_ERR_WORKSPACE;
    hipStream_t st = (hipStream_t) stream;
    const int64_t n_len = mi355x_log_mel_n_len(n_samples);
    int64_t n_frames = (n_samples + MEL_NFFT / 2) / MEL_HOP + 1;
    if (n_frames > n_len) n_frames = n_len;
    const int64_t rounds = (n_frames + MEL_FRAMES - 1) / MEL_FRAMES;
    const int64_t per_group = (rounds + MEL_GROUPS - 1) / MEL_GROUPS, groups = (rounds + per_group - 1) / per_group;
    const int64_t gx = (n_len + 256 * MEL_FINISH - 1) / (256 * MEL_FINISH);
    if (gx > 0x7fffffff) return MI355X_ERR_UNSUPPORTED;
    float * maxima = (float *) workspace;
    k_log_mel_frames<<<(unsigned) groups, 256, 0, st>>>(samples, n_samples, filters, n_mel, n_frames, n_len, per_group, mel, maxima);
    if (const int rc = launch_status()) return rc;
    k_log_mel_finish<<<dim3((unsigned) gx, (unsigned) n_mel), 256, 0, st>>>(mel, n_frames, n_len, maxima, (int) groups);
    return launch_status();
}
