// Internal interface of the learned warm start (learn.hip): the neighbour
// features, the 64 -> 128 -> 128 -> 2 SiLU network on bf16 MFMA, its
// training kernels and Adam.  Not installed; the public ABI is wrach.h.
#pragma once

#include "frame.h"

namespace wrach {

constexpr int kNbrs = 16;     // neighbours per particle
constexpr int kFeat = 64;     // kNbrs x (dx, dy, dvx, dvy)
constexpr int kHid = 128;     // hidden width of both layers
constexpr int kOutDim = 2;    // predicted displacement (dx, dy)
// Most particles in a particle's 5x5 cells for it to get features (else
// all-zero features): a bound on one lane's work, as kStencilBudget is for
// the 3x3 cells of a separation pass.
constexpr uint32_t kFeatBudget = 4096;

// The master parameters, f32, in one vector: W1[64][128] (input-major),
// b1[128], W2[128][128], b2[128], W3[128][2], b3[2].
constexpr uint32_t kOffW1 = 0;
constexpr uint32_t kOffB1 = kOffW1 + kFeat * kHid;
constexpr uint32_t kOffW2 = kOffB1 + kHid;
constexpr uint32_t kOffB2 = kOffW2 + kHid * kHid;
constexpr uint32_t kOffW3 = kOffB2 + kHid;
constexpr uint32_t kOffB3 = kOffW3 + kHid * kOutDim;
constexpr uint32_t kParams = kOffB3 + kOutDim;

// The dense layers' weights as v_mfma_f32_16x16x32_bf16 A operands: a
// fragment is 64 lanes x 8 bf16 (1 KiB), lane l holding row 16t + l % 16 of
// a 16-row tile t and the 8 entries of k-step s that its lane group l / 16
// supplies.  W1 (A = W1^T, rows = outputs): 8 x 2 fragments; W2 forward
// (A = W2^T): 8 x 4; W2 backward (A = W2, rows = inputs): 8 x 4.
constexpr uint32_t kFragElems = 512;
constexpr uint32_t kW1Frags = (kHid / 16) * (kFeat / 32);
constexpr uint32_t kW2Frags = (kHid / 16) * (kHid / 32);
constexpr uint32_t kFragW1 = 0;
constexpr uint32_t kFragW2F = kFragW1 + kW1Frags;
constexpr uint32_t kFragW2B = kFragW2F + kW2Frags;
constexpr uint32_t kFrags = kFragW2B + kW2Frags;

// Packed weights the kernels read: fragments (bf16 bits), W3 rounded to
// bf16 and held as f32, and the f32 master vector (biases).
struct MlpWeights {
    const uint16_t *frag;  // kFrags * kFragElems
    const float *w3;       // [128][2]
    const float *params;   // kParams
};

// Neighbour features of the packed state (pos, vel) for particles
// [0, p.n): row row0 + i of `feat` (64 bf16) for particle i.  Optional:
// what the separation passes that follow need, in their lane order (`perm`,
// null: the particles' own) -- the rows of each lane's 3x3 cells (`rows`,
// `rows2`), or without them each particle's cell (`cell`), and the budget's
// word (`words`) -- and the overlap sums of these positions over the 3x3
// cells as a separation pass measures them, added to `sums` (the layout of
// the stencil sums: slot block % kStencilSumSlots).
struct FeatureArgs {
    const float2 *pos;
    const float2 *vel;
    float4 *state;  // workspace: (pos, vel) of each particle (null: gathered apart)
    uint16_t *feat;
    uint32_t row0;
    const uint32_t *perm;
    uint4 *rows;
    uint2 *rows2;
    uint32_t *cell;
    uint32_t *words;
    unsigned long long *sums;
};
hipError_t launch_learn_features(const FrameParams &p, const FrameBuffers &b, const FeatureArgs &a,
                                 hipStream_t stream);

// Inference over rows [0, n) of `feat`: y_out[i] = the network's output
// (if not null); pout[i] = pin[i] + clamp(y, +-kMaxWarm) (if not null).
constexpr float kMaxWarm = 1.0f;
struct InferArgs {
    const uint16_t *feat;
    uint32_t n;
    float2 *y_out;
    const float2 *pin;
    float2 *pout;
};
hipError_t launch_learn_infer(const MlpWeights &w, const InferArgs &a, hipStream_t stream);
// Blocks of the inference kernel the device holds at once.
uint32_t resident_blocks_infer();

// One training step's buffers (batch rows bsz, a multiple of 64).
constexpr uint32_t kWeights = kFeat * kHid + kHid * kHid;  // dW1 and dW2 of a chunk
constexpr uint32_t kCols = 4 * kHid + 3;                   // b1, b2, W3, b3, squared error
struct TrainArgs {
    const uint16_t *feat;    // training rows
    const float2 *target;    // their targets
    const uint32_t *sel;     // batch row p is training row sel[p]
    uint32_t bsz;
    float inv_bsz;           // 1 / bsz
    // The weight gradients' k chunks: `chunks` of kc rows, a multiple of 32
    // (the last one possibly shorter).
    uint32_t kc, chunks;
    // Activations and gradients, per 16 batch rows [feature][16]:
    uint16_t *xt;            // 64 features: the inputs
    uint16_t *a1t, *dz1t;    // 128: SiLU(z1), dL/dz1 (bf16)
    uint16_t *dz2t;          // 128: dL/dz2 (bf16)
    float *a2t;              // 128: SiLU(z2)
    float *dyt;              // [2][bsz] dL/dy
    float *sqerr;            // [bsz / 16] squared error per 16 rows
    float *part;             // [chunks][kWeights]
    float *cols;             // [kCols] column sums
};
// part and cols.
hipError_t launch_learn_grad(const MlpWeights &w, const TrainArgs &a, hipStream_t stream);
// The gradient from part and cols, or `given`; with `grad` it is written
// there, otherwise Adam on the master vector (f32, in place) and the packed
// weights.
struct UpdateArgs {
    const float *part;
    const float *cols;
    uint32_t chunks;
    const float *given;
    float *loss;        // loss_scale * the sum of squared errors (if not null)
    float loss_scale;
    float *grad;
    float *params, *m, *v;
    uint16_t *frag;
    float *w3;
    float lr, beta1, beta2, eps;
    float c1, c2;  // 1 / (1 - beta1^t), 1 / (1 - beta2^t)
};
hipError_t launch_learn_update(const UpdateArgs &u, hipStream_t stream);
hipError_t launch_learn_pack(const float *params, uint16_t *frag, float *w3, hipStream_t stream);
// target[row0 + i] = pk[i] - p0[i] for i < n.
hipError_t launch_learn_target(const float2 *pk, const float2 *p0, float2 *target, uint32_t row0,
                               uint32_t n, hipStream_t stream);

}  // namespace wrach
