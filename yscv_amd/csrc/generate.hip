// Host-side sampling loop over the device-resident decoder: the counterpart of generate() / sample_token()
// (crates/yscv-onnx/src/generate.rs:58-208).  The reference re-runs its model on the whole sequence for every
// token; here every token is one decode step against the KV cache, the logits of that step come back to the host
// and the reference's sampler runs on them operation by operation (repetition penalty, temperature, top-k
// threshold, softmax, top-p cut, xorshift64 draw).  Greedy decoding (top_k = 1 with no ties) gives the tokens
// yscv_hip_decoder_run picks on the device.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <functional>
#include <numeric>
#include <vector>

#include "common.hpp"

using namespace yscv;

namespace {

// f32::max(a, b): a NaN operand is ignored
inline float rust_max(float a, float b) { return (b != b) ? a : ((a != a) ? b : (a > b ? a : b)); }

// indices sorted by descending value; incomparable (NaN) pairs count as equal (generate.rs:128-133, 160-165).
// The reference uses an unstable sort, so the order among equal values is unspecified there; a stable sort fixes it
// to ascending index here.
std::vector<size_t> sorted_desc(const float *v, size_t n) {
  std::vector<size_t> idx(n);
  std::iota(idx.begin(), idx.end(), (size_t)0);
  std::stable_sort(idx.begin(), idx.end(), [&](size_t a, size_t b) { return v[a] > v[b]; });
  return idx;
}

// The whole of sample_token on full sorts, as the reference writes it: what logits with a NaN or +inf among them take
// (their order is whatever the sort makes of incomparable pairs).  Every other input goes through sample_selected.
uint32_t sample_sorted(float *logits, size_t vocab_size, size_t top_k, float top_p, float u) {
  // top-k: everything below the k-th largest logit is removed (generate.rs:125-141)
  if (top_k > 0 && top_k < vocab_size) {
    const std::vector<size_t> order = sorted_desc(logits, vocab_size);
    const float threshold = logits[order[top_k - 1]];
    for (size_t i = 0; i < vocab_size; i++)
      if (logits[i] < threshold) logits[i] = -INFINITY;
  }
  // softmax (generate.rs:143-155)
  float max_val = -INFINITY;
  for (size_t i = 0; i < vocab_size; i++) max_val = rust_max(max_val, logits[i]);
  float sum = 0.0f;
  for (size_t i = 0; i < vocab_size; i++) {
    logits[i] = expf(logits[i] - max_val);
    sum += logits[i];
  }
  if (sum > 0.0f) {
    const float inv = 1.0f / sum;
    for (size_t i = 0; i < vocab_size; i++) logits[i] *= inv;
  }
  // top-p: keep the most probable tokens until their cumulative probability exceeds p (generate.rs:157-186)
  if (top_p < 1.0f) {
    const std::vector<size_t> order = sorted_desc(logits, vocab_size);
    float cumsum = 0.0f;
    for (size_t pos = 0; pos < vocab_size; pos++) {
      cumsum += logits[order[pos]];
      if (cumsum > top_p) {
        for (size_t rest = pos + 1; rest < vocab_size; rest++) logits[order[rest]] = 0.0f;
        break;
      }
    }
    float new_sum = 0.0f;
    for (size_t i = 0; i < vocab_size; i++) new_sum += logits[i];
    if (new_sum > 0.0f) {
      const float inv = 1.0f / new_sum;
      for (size_t i = 0; i < vocab_size; i++) logits[i] *= inv;
    }
  }
  float cumsum = 0.0f;
  for (size_t i = 0; i < vocab_size; i++) {
    cumsum += logits[i];
    if (cumsum > u) return (uint32_t)i;
  }
  // fallback: the most probable token; Iterator::max_by keeps the last of equal maxima (generate.rs:202-207)
  size_t best = 0;
  for (size_t i = 1; i < vocab_size; i++)
    if (!(logits[best] > logits[i])) best = i;
  return (uint32_t)best;
}

constexpr size_t kBlock = 64;        // values a compare-and-skip test covers: one vector loop without a branch inside
constexpr size_t kHeapMaxK = 1024;   // above this many kept logits a heap insertion costs more than a selection pass

// the k-th largest of v[0 .. n), 1 <= k <= n, no NaN
float kth_largest(const float *v, size_t n, size_t k) {
  if (k > kHeapMaxK) {
    std::vector<float> copy(v, v + n);
    std::nth_element(copy.begin(), copy.begin() + (k - 1), copy.end(), std::greater<float>());
    return copy[k - 1];
  }
  // min-heap of the k largest so far; a block without a value above the heap's smallest is skipped whole
  std::vector<float> heap(v, v + k);
  std::make_heap(heap.begin(), heap.end(), std::greater<float>());
  auto offer = [&](float x) {
    if (x > heap.front()) {
      std::pop_heap(heap.begin(), heap.end(), std::greater<float>());
      heap.back() = x;
      std::push_heap(heap.begin(), heap.end(), std::greater<float>());
    }
  };
  size_t i = k;
  for (; i + kBlock <= n; i += kBlock) {
    const float lo = heap.front();
    int any = 0;
    for (size_t j = 0; j < kBlock; j++) any |= v[i + j] > lo;
    if (any)
      for (size_t j = 0; j < kBlock; j++) offer(v[i + j]);
  }
  for (; i < n; i++) offer(v[i]);
  return heap.front();
}

// keys[from ..) in ascending order.  The high halves are sorted 11 bits at a time; the low halves (indices) are put in
// order first, so equal high halves keep ascending indices.
void radix_sort_high32(std::vector<uint64_t> &keys, size_t from) {
  std::vector<uint64_t> tmp(keys.size() - from);
  uint64_t *a = keys.data() + from, *b = tmp.data();
  const size_t n = tmp.size();
  for (int shift : {0, 11, 22, 32, 43, 54}) {
    const uint64_t mask = shift == 22 || shift == 54 ? 0x3FF : 0x7FF;
    size_t count[2048] = {0};
    for (size_t i = 0; i < n; i++) count[(a[i] >> shift) & mask]++;
    size_t at = 0;
    for (size_t &c : count) {
      const size_t here = c;
      c = at;
      at += here;
    }
    for (size_t i = 0; i < n; i++) b[count[(a[i] >> shift) & mask]++] = a[i];
    std::swap(a, b);
  }  // six passes: the result is back in keys
}

// sample_token for logits without NaN or +inf and at least one finite: same operations in the same order as
// sample_sorted on every value that matters, without the sorts.  A logit below the top-k threshold becomes a
// probability of exactly 0, and adding 0 changes none of the sums, so all passes after the threshold run over the
// kept indices only (ascending); the top-p cut looks at the most probable ones in a growing selected prefix.
// Two full sorts of a 151 936-token vocabulary take 15 ms; the selection takes 0.05 .. 0.1 ms with top_k = 50.
uint32_t sample_selected(float *logits, size_t vocab_size, size_t top_k, float top_p, float u) {
  std::vector<uint32_t> kept;
  if (top_k > 0 && top_k < vocab_size) {
    const float threshold = kth_largest(logits, vocab_size, top_k);
    kept.reserve(2 * top_k);
    size_t i = 0;
    for (; i + kBlock <= vocab_size; i += kBlock) {
      int any = 0;
      for (size_t j = 0; j < kBlock; j++) any |= logits[i + j] >= threshold;
      if (any)
        for (size_t j = 0; j < kBlock; j++)
          if (logits[i + j] >= threshold) kept.push_back((uint32_t)(i + j));
    }
    for (; i < vocab_size; i++)
      if (logits[i] >= threshold) kept.push_back((uint32_t)i);
  } else {
    kept.resize(vocab_size);
    std::iota(kept.begin(), kept.end(), 0u);
  }
  std::vector<float> p(kept.size());
  float max_val = -INFINITY;
  for (size_t j = 0; j < kept.size(); j++) {
    p[j] = logits[kept[j]];
    max_val = p[j] > max_val ? p[j] : max_val;
  }
  float sum = 0.0f;
  for (float &v : p) {
    v = expf(v - max_val);
    sum += v;
  }
  float inv = 1.0f / sum;  // the largest term is 1
  for (float &v : p) v *= inv;
  std::memset(logits, 0, vocab_size * sizeof(float));
  if (top_p < 1.0f) {
    // Positions in p by descending probability, ascending index among equals, as one integer key each (probabilities
    // are not negative, so their bit patterns order like the values).  A peaked distribution is cut within the first
    // few hundred: two selected prefixes; a flat one is radix-sorted whole.
    std::vector<uint64_t> order(p.size());
    for (size_t j = 0; j < p.size(); j++) {
      uint32_t bits;
      std::memcpy(&bits, &p[j], 4);
      order[j] = ((uint64_t)~bits << 32) | j;
    }
    float cumsum = 0.0f;
    bool cut = false;
    size_t done = 0;
    for (size_t want = 64; done < p.size() && !cut; want *= 8) {
      size_t end = p.size();
      if (want <= 512 && want < p.size() - done) {
        end = done + want;
        std::nth_element(order.begin() + done, order.begin() + end, order.end());
      }
      if (end - done > 2048) radix_sort_high32(order, done);
      else std::sort(order.begin() + done, order.begin() + end);
      for (; done < end; done++) {
        cumsum += p[(uint32_t)order[done]];
        if (cumsum > top_p) {
          done++;
          cut = true;
          break;
        }
      }
    }
    for (size_t j = done; j < order.size(); j++) p[(uint32_t)order[j]] = 0.0f;  // nothing is left when no cut was reached
    float new_sum = 0.0f;
    for (float v : p) new_sum += v;
    if (new_sum > 0.0f) {
      inv = 1.0f / new_sum;
      for (float &v : p) v *= inv;
    }
  }
  for (size_t j = 0; j < p.size(); j++) logits[kept[j]] = p[j];
  float cumsum = 0.0f;
  for (size_t j = 0; j < p.size(); j++) {
    cumsum += p[j];
    if (cumsum > u) return kept[j];
  }
  size_t best = 0;
  for (size_t j = 1; j < p.size(); j++)
    if (!(p[best] > p[j])) best = j;
  return kept[best];
}

// xorshift64 draw (generate.rs:188-192); `u64 as f32` rounds to nearest, u64::MAX as f32 is 2^64
float draw(uint64_t *rng) {
  uint64_t x = *rng;
  x ^= x << 13;
  x ^= x >> 7;
  x ^= x << 17;
  *rng = x;
  return (float)x / 18446744073709551616.0f;
}

}  // namespace

namespace yscv {
int32_t decoder_top_candidates(yscv_hip_decoder *d, size_t k, float scale, std::vector<float> &values, std::vector<uint32_t> &indices,
                               bool *whole);
}

extern "C" {

int32_t yscv_hip_sample_token(float *logits, size_t vocab_size, size_t top_k, float top_p, uint64_t *rng, uint32_t *token_out) {
  YSCV_REQUIRE(logits && rng && token_out, "null argument");
  YSCV_REQUIRE(vocab_size > 0, "empty vocabulary");
  const float u = draw(rng);
  int odd = 0, finite = 0;  // a NaN or +inf anywhere; anything above -inf anywhere
  for (size_t i = 0; i < vocab_size; i++) {
    odd |= !(logits[i] <= FLT_MAX);
    finite |= logits[i] >= -FLT_MAX;
  }
  *token_out = (odd || !finite || vocab_size > UINT32_MAX) ? sample_sorted(logits, vocab_size, top_k, top_p, u)
                                                           : sample_selected(logits, vocab_size, top_k, top_p, u);
  return YSCV_HIP_OK;
}

int32_t yscv_hip_decoder_generate(yscv_hip_decoder *d, const uint32_t *input_ids, size_t n_input,
                                  const yscv_hip_generate_config *cfg, uint32_t *generated_out, size_t *n_generated) {
  YSCV_REQUIRE(d && input_ids && cfg && n_generated, "null argument");
  YSCV_REQUIRE(n_input > 0, "empty prompt");
  YSCV_REQUIRE(cfg->max_tokens == 0 || generated_out != nullptr, "null output buffer");
  *n_generated = 0;
  size_t vocab = 0;
  YSCV_TRY(yscv_hip_decoder_vocab(d, &vocab));
  std::vector<uint32_t> tokens(input_ids, input_ids + n_input);
  std::vector<float> logits(vocab);
  uint64_t rng_state = 0xdeadbeefULL;  // generate.rs:68
  // the prompt goes through the decoder in one pass (yscv_hip_decoder_prefill: every projection sees all positions at
  // once); the KV cache then holds positions 0 .. n_input-1 and the logits are those of the last prompt position
  {
    std::vector<int32_t> prompt(n_input);
    for (size_t p = 0; p < n_input; p++) {
      YSCV_REQUIRE(input_ids[p] < vocab, "prompt token %u outside the vocabulary (%zu)", input_ids[p], vocab);
      prompt[p] = (int32_t)input_ids[p];
    }
    YSCV_REQUIRE(n_input < ((size_t)1 << 31), "prompt too long");
    YSCV_TRY(yscv_hip_decoder_prefill(d, prompt.data(), (int32_t)n_input, 0, nullptr));
  }
  const bool scaled = cfg->temperature != 1.0f && cfg->temperature > 0.0f;
  const float inv_temp = scaled ? 1.0f / cfg->temperature : 1.0f;
  std::vector<float> cand;
  std::vector<uint32_t> cand_index;
  for (size_t g = 0; g < cfg->max_tokens; g++) {
    // Without a repetition penalty the device sends the few logits that top-k can keep (multiplied by 1 / temperature there,
    // the same f32 product): everything below the k-th largest has probability 0 in sample_token, so the sampler gives the
    // same token on those alone.  A sampled token of a 151936-token vocabulary beside prompt and decode steps: 100 -> 3 us.
    bool whole = true;
    uint32_t next = 0;
    if (cfg->repetition_penalty == 1.0f && inv_temp > 0.0f && inv_temp <= FLT_MAX && cfg->top_k < vocab)
      YSCV_TRY(decoder_top_candidates(d, cfg->top_k, inv_temp, cand, cand_index, &whole));
    if (!whole) {
      const float u = draw(&rng_state);
      next = cand_index[sample_selected(cand.data(), cand.size(), cfg->top_k, cfg->top_p, u)];
    }
    if (whole) YSCV_TRY(yscv_hip_decoder_read_logits(d, logits.data()));
    if (whole && cfg->repetition_penalty != 1.0f) {  // generate.rs:80-92
      for (uint32_t t : tokens) {
        if (t < logits.size()) {
          if (logits[t] > 0.0f) logits[t] /= cfg->repetition_penalty;
          else logits[t] *= cfg->repetition_penalty;
        }
      }
    }
    if (whole && scaled) {  // generate.rs:95-100
      for (float &v : logits) v *= inv_temp;
    }
    if (whole) YSCV_TRY(yscv_hip_sample_token(logits.data(), vocab, cfg->top_k, cfg->top_p, &rng_state, &next));
    if (cfg->has_eos && cfg->eos_token_id == next) break;
    generated_out[(*n_generated)++] = next;
    tokens.push_back(next);
    if (g + 1 == cfg->max_tokens) break;
    const int32_t tok = (int32_t)next;
    YSCV_TRY(yscv_hip_decoder_reset(d, 1, (int32_t)(tokens.size() - 1), &tok));
    YSCV_TRY(yscv_hip_decoder_run(d, 1, YSCV_HIP_DECODE_AUTO, nullptr));
  }
  return YSCV_HIP_OK;
}

}  // extern "C"
