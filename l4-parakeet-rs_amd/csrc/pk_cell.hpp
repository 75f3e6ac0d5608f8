// The long form's LSTM cell in IEEE basic operations (fma, division, rounding,
// scaling by powers of two), so that the INT8 roundings of its outputs, which
// amplify one ulp into a different token, are reproduced bit for bit by a CPU
// evaluating the same operations.  Host and device compile the same functions.
//
// The quotients are divisions.  One Newton step on the hardware reciprocal
// equals them only where the reciprocal's seed allows it (a seed one ulp off
// the rounded value gives a wrong last bit for 1 or 31 mantissas), and with
// the branch that its range needs it was slower: the general kernel at H = 512,
// 1024 frames, 9.10 against 8.94 ms, the 640 kernel, 7500 frames, 42.1 / 41.8.
#pragma once

#pragma clang force_cuda_host_device begin

namespace pk {

// exp(x) from IEEE basic operations only, so that the long form's cell (whose
// outputs are rounded to INT8) is reproduced bit for bit by a CPU evaluating
// the same operations: Cody-Waite reduction x = n ln2 + r (ln2 split into a
// 16-bit head, so n * head is exact, and a tail), e^r by its degree-7 Taylor
// polynomial (|r| <= 0.347: truncation error 5e-9 relative), times 2^n.
// Within 0.82 ulp of exp over [-87, 88]; expf / tanhf of the reference are
// within about an ulp too.
inline float det_exp(float x) {
    if (x != x) return x;
    x = __builtin_fminf(__builtin_fmaxf(x, -104.0f), 89.0f);
    const float n = __builtin_rintf(x * 1.44269504f);
    float r = __builtin_fmaf(n, -0.693145751953125f, x);
    r = __builtin_fmaf(n, -1.428606765330187e-06f, r);
    float q = 1.98412698e-04f;
    q = __builtin_fmaf(q, r, 1.38888889e-03f);
    q = __builtin_fmaf(q, r, 8.33333333e-03f);
    q = __builtin_fmaf(q, r, 4.16666667e-02f);
    q = __builtin_fmaf(q, r, 1.66666667e-01f);
    q = __builtin_fmaf(q, r, 0.5f);
    q = __builtin_fmaf(q, r, 1.0f);
    q = __builtin_fmaf(q, r, 1.0f);
    return __builtin_ldexpf(q, (int)n);
}
inline float det_sigmoid(float v) { return 1.0f / (1.0f + det_exp(-v)); }
// tanh(x) = sign(x) (1 - e^-2|x|) / (1 + e^-2|x|): absolute error ~1e-7.
inline float det_tanh(float v) {
    const float t = det_exp(-2.0f * __builtin_fabsf(v));
    return __builtin_copysignf((1.0f - t) / (1.0f + t), v);
}
// det_tanh(v) for the cell gate, det_sigmoid(v) for the others, with one
// exponential and one division: lanes of one wave evaluate different gates.
inline float det_gate(float v, bool cell) {
    const float e = det_exp(cell ? -2.0f * __builtin_fabsf(v) : -v);
    const float q = (cell ? 1.0f - e : 1.0f) / (1.0f + e);
    return cell ? __builtin_copysignf(q, v) : q;
}

// decoder.cu:116-129 lstm_cell with the transcendental functions above; the
// cell update is fma(f, c, i * g).
inline void lstm_cell(const float (&s)[4], float c_prev, float& c_out, float& h_out) {
    const float ig = det_sigmoid(s[0]), fg = det_sigmoid(s[1]), cg = det_tanh(s[2]), og = det_sigmoid(s[3]);
    c_out = __builtin_fmaf(fg, c_prev, ig * cg);
    h_out = og * det_tanh(c_out);
}

}  // namespace pk

#pragma clang force_cuda_host_device end
