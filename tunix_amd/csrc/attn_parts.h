// What a decode step's attention leaves where the key range is cut into chunks (attention.hip), for whatever merges them: of query vector v and chunk
// c, from ws + (v n_chunks + c)(head_dim + kPartPad) on, the running maximum m, the sum l of exponentials under it, two numbers of no meaning and
// O[head_dim]; out = sum_c e^{m_c - M} O_c / sum_c e^{m_c - M} l_c.  A chunk without a key has l = 0 and an O that nobody wrote; l is 0, positive, or the
// NaN of a query or a key, which has to reach the output.
#pragma once

namespace {
constexpr float kNegBig = -1.0e30f;
constexpr int kPartPad = 4;   // keeps O on 16 bytes
}  // namespace
