// Library-internal fused nn op, for the GPT forward.
#pragma once

#include <stddef.h>

namespace bmb {

// res_out = a + b (residual_forward), then ln_out, mean, rstd =
// layernorm(res_out) (layernorm_forward), in one pass over the rows: the same
// fp32 results as the two launches of src/gpt.cu:266-268,278-283. Null stream.
void residual_layernorm_forward(float *res_out, float *ln_out, float *mean, float *rstd,
                                const float *a, const float *b, const float *weight,
                                const float *bias, int N, int C);

// Column sums in two steps, for the GPT backward: partial sums over groups of
// rows that the kernels producing (or reading) a gradient leave behind, and one
// launch that finishes several of them. A job's partial is G rows of
// n[0] + n[1] + n[2] columns; column sums are added onto dst[0][0..n[0]),
// then dst[1], then dst[2]. Null stream; every sum in a fixed order.
struct ColsumJob {
    const float *partial;
    float *dst[3];
    int n[3];
    int G;
};
constexpr int COLSUM_JOBS = 6;
void colsum_finish_jobs(const ColsumJob *jobs, int count);  // count <= COLSUM_JOBS

// bias_backward up to its finish: partial holds bias_partial_floats(N, C).
size_t bias_partial_floats(int N, int C);
ColsumJob bias_backward_partial(float *dbias, const float *dout, int N, int C, float *partial);

// layernorm_backward up to its finish, with (dsum not null) the column sums of
// the updated dinp added onto dsum as bias_backward(dsum, dinp, N, C) would.
// partial holds layernorm_partial_floats(N, C). Returns false where a row does
// not fit the fused kernel: everything is then done, with no job left.
size_t layernorm_partial_floats(int N, int C);
bool layernorm_backward_partial(float *dinp, float *dweight, float *dbias, float *dsum,
                                const float *dout, const float *inp, const float *weight,
                                const float *mean, const float *rstd, int N, int C,
                                float *partial, ColsumJob &job);

}  // namespace bmb
