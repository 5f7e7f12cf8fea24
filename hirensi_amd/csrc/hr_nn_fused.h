/* Learned gradient preconditioner: calls that fuse steps of hirensi_nn.h the
 * network takes together (internal to the package: hirensi_amd/precond.py calls
 * them).  Same conventions (device pointers, work queued on
 * `stream`, 0 or a nonzero error code); each equals its parts bit for bit.
 */
#ifndef HR_NN_FUSED_H
#define HR_NN_FUSED_H

#ifdef __cplusplus
extern "C" {
#endif

/* hr_nn_conv3d with what follows it in a network: + add (may be NULL, may be
 * out), then leaky ReLU of the given slope (1: none), or, where gate (an
 * activation output of out's shape) is given, the leaky ReLU's backward:
 * out = gate > 0 ? s : slope s. */
int hr_nn_conv3d_fused(const float* in, const unsigned short* w, const float* bias, const float* add,
                       const float* gate, float slope, float* out, int cin, int cout, int NB, int D, int H, int W,
                       void* stream);

/* hr_nn_transpose_weights of nlayer (<= 32) layers whose weights follow one
 * another in w and wt; cin, cout are host arrays. */
int hr_nn_transpose_layers(const unsigned short* w, unsigned short* wt, int nlayer, const int* cin, const int* cout,
                           void* stream);

/* The pooling backward added to dx, then the leaky ReLU's backward at its output y
 * (the shape of dx). */
int hr_nn_avgpool2_grad_act(const float* dy, const float* y, float* dx, long long C, int D, int H, int W, float slope,
                            void* stream);

/* The upsampling backward, then the leaky ReLU's backward at its output y (the
 * coarse shape; NULL: none). */
int hr_nn_upsample2_grad_act(const float* dy, const float* y, float* dx, long long C, int D, int H, int W, float slope,
                             void* stream);

#ifdef __cplusplus
}
#endif

#endif
