// Kernels of the learned initial guess (a 3D U-Net on node-centred grids, channels-last bf16
// tensors, fp32 accumulation on the matrix cores).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace sr {

typedef uint16_t bf16_t;   // bfloat16 bit pattern

// grid of one network level: node counts and the 4 x 4 x 16 output tiles of the convolutions
struct NetGrid {
    int nx, ny, nz;
    int tx, ty, tz;   // tile counts
    __host__ __device__ long nvox() const { return (long)nx * ny * nz; }
    __host__ __device__ long ntiles() const { return (long)tx * ty * tz; }
};

// t = q n + r and t = (i n1 + j) n2 + k: in 32 bits where t has no more (64-bit divisions cost some hundred
// instructions each)
__device__ inline void split2(long t, int n, long &q, int &r) {
    if (t >> 32) {
        q = t / n;
        r = (int)(t - q * n);
    } else {
        const unsigned u = (unsigned)t, a = u / (unsigned)n;
        q = a;
        r = (int)(u - a * (unsigned)n);
    }
}
__device__ inline void node3(long t, int n1, int n2, int &i, int &j, int &k) {
    long a, b;
    split2(t, n2, a, k);
    split2(a, n1, b, j);
    i = (int)b;
}

inline NetGrid net_grid(int nx, int ny, int nz) {
    NetGrid g{nx, ny, nz, (nx + 3) / 4, (ny + 3) / 4, (nz + 15) / 16};
    return g;
}

enum ConvOut { CONV_BF16_RELU = 0, CONV_F32 = 1, CONV_F32_CH0 = 2, CONV_MASK = 3 };

// packed-weight size (bf16 elements) of a convolution CIN -> COUT
long conv_pack_elems(int cin, int cout);
// W (27, COUT, CIN) fp32 master weights -> packed bf16 fragments of the convolution; with
// transpose, the packing of the adjoint convolution (COUT -> CIN, taps mirrored).  Any number of
// layers in one launch: workgroups first[q] to first[q + 1] - 1 take segment q.
constexpr int kMaxSegs = 24;   // two for each layer
struct PackSegs {
    int n = 0, first[kMaxSegs + 1] = {};
    const float *W[kMaxSegs];
    bf16_t *packed[kMaxSegs];
    int cin[kMaxSegs], cout[kMaxSegs], transpose[kMaxSegs];
    long total[kMaxSegs];
};
void add_pack(PackSegs &P, const float *W, int cin, int cout, int transpose, bf16_t *packed);
void launch_pack(const PackSegs &P, hipStream_t s);
// out = conv(in) (+ bias, ReLU, bf16), raw fp32, or (CONV_MASK) bf16(conv(in) * (act > 0)).  At 129^3 x 16
// channels the gradient through a ReLU as fp32 and a second kernel took 71 + 98 us, 74 this way.
int launch_conv(int cin, int cout, const NetGrid &g, const bf16_t *in, const bf16_t *wpack, const float *bias,
                void *out, int mode, const bf16_t *act, hipStream_t s);
// weight gradient: partials per slot, then the fixed-order sum into dW (27, COUT, CIN) fp32
int wgrad_slots(int cin, int cout, const NetGrid &g);
long wgrad_part_elems(int cin, int cout, const NetGrid &g);
// with bpart (wgrad_slots x cout floats) the bias gradient db (cout) of the same output gradient
// comes from the same pass: the blocks of input block 0 add the staged gradient tiles per channel
int launch_wgrad(int cin, int cout, const NetGrid &g, const bf16_t *dy, const bf16_t *x, float *part, float *dW,
                 float *bpart, float *db, hipStream_t s);
// transfer operators on channels-last tensors (C a multiple of 4)
void launch_restrict_bf16(const NetGrid &fine, const NetGrid &coarse, int C, const bf16_t *in, bf16_t *out,
                          hipStream_t s);
// out = bf16(scale R(in) * (act > 0))
void launch_restrict_mask(const NetGrid &fine, const NetGrid &coarse, int C, const float *in, const bf16_t *act,
                          bf16_t *out, float scale, hipStream_t s);
// out = bf16(P(coarse) + skip)
void launch_prolong_add_bf16(const NetGrid &fine, const NetGrid &coarse, int C, const bf16_t *coarse_in,
                             const bf16_t *skip, bf16_t *out, hipStream_t s);
// out = bf16((acc + scale P(coarse)) * (act > 0)), the sum in fp32
void launch_prolong_add_mask(const NetGrid &fine, const NetGrid &coarse, int C, const float *coarse_in,
                             const float *acc, const bf16_t *act, bf16_t *out, float scale, hipStream_t s);
void launch_f32_to_bf16(long n, const float *in, bf16_t *out, hipStream_t s);
void launch_bf16_to_f32(long n, const bf16_t *in, float *out, hipStream_t s);
// one channel of dy into a 16-channel bf16 tensor (the other channels zero)
void launch_expand_ch0(long nvox, const float *dy, bf16_t *out16, hipStream_t s);
// Adam on fp32 master weights (bias-corrected step sizes given by the host), segments as in PackSegs: the
// step of all layers took 47 launches with its packing, 480 us, and takes two
struct AdamSegs {
    int n = 0, first[kMaxSegs + 1] = {};
    float *w[kMaxSegs];
    const float *g[kMaxSegs];
    float *m[kMaxSegs], *v[kMaxSegs];
    int count[kMaxSegs];
};
void add_adam(AdamSegs &A, int n, float *w, const float *g, float *m, float *v);
void launch_adam(const AdamSegs &A, float lr_t, float beta1, float beta2, float eps, hipStream_t s);

}  // namespace sr
