// Host placement planner at world = 1.
//
// Reference: ferry/policy.py:130-194 (plan_layer), :109-127 (_choose_slot), :197-205
// (layer_slots), :36-46 (_admission_capacity) and the quota check of ferry/quota.py:63.
// At world = 1 both the FERRY and the RANDOM policy assign every miss to rank 0 (the quota
// table row is [m] and randint(0, 1) is 0), so only the capacity check, the slot choice and
// the state update remain.  The eviction key is the lexicographic minimum of
// (fp32 score of the key's own layer, last-use tick, key) over slots that do not hold an
// expert the current layer needs; the first empty slot wins outright.  ferry_choose_slot is
// that rule for one miss; a layer call applies it to all of its misses through one partial
// sort of the slots (the same choices, see plan_demand).  The call's routing IDs are scanned
// once, which validates them and counts each expert's demand (returned by ferry_plan_fetch); of a
// large call the device does both (ferry_history_count) and the planner sums its records: the scan
// of 65,536 tokens x 6 IDs took 348 us, of 8192 x 8 about 60 us, with the GPU waiting.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "../../include/ferry_amd.h"
#include "count_records.h"

namespace ferry {
void set_error(const char* fmt, ...);
void clear_error();
}  // namespace ferry

extern "C" int64_t ferry_choose_slot(int64_t layer, const uint8_t* active, const int64_t* slots,
                                     int64_t cap, const int64_t* last, const float* scores,
                                     int64_t experts) {
  // same initial key as the reference: (inf, 2^60, 2^60); scores widen exactly to double
  int64_t best = -1;
  double best_score = __builtin_inf();
  int64_t best_used = (int64_t)1 << 60, best_key = (int64_t)1 << 60;
  for (int64_t i = 0; i < cap; ++i) {
    const int64_t key = slots[i];
    if (key < 0) return i;
    if (key / experts == layer && active[key % experts]) continue;  // needed by this layer
    const double score = scores[key];
    const int64_t used = last[key];
    if (score < best_score ||
        (score == best_score && (used < best_used || (used == best_used && key < best_key)))) {
      best = i;
      best_score = score;
      best_used = used;
      best_key = key;
    }
  }
  return best;
}

namespace {

// Demand scan over routing IDs of type T (int64 from the Python API, uint8 from the mapped
// staging buffer): one pass validates them (every ID in [0, E), none repeated within a token:
// the reference's demand count and layout assume both) and counts each expert's demand.
// 0, or -3 with the error set.
template <typename T>
int64_t scan_ids(const T* ids, int64_t tokens, int64_t topk, int64_t experts,
                 std::vector<int64_t>* demand, const char* who) {
  // Four demand histograms, by token mod 4, so that consecutive tokens naming the same expert
  // do not chain their increments through one memory word; a token's repeated IDs are found
  // with a per-expert last-token array.
  std::vector<int64_t> hist((size_t)(4 * experts), 0);
  std::vector<int32_t> seen((size_t)experts, -1);
  for (int64_t t = 0; t < tokens; ++t) {
    const T* row = ids + t * topk;
    int64_t* h = hist.data() + (t & 3) * experts;
    const int32_t tt = (int32_t)t;
    for (int64_t j = 0; j < topk; ++j) {
      const int64_t e = (int64_t)row[j];
      if (e < 0 || e >= experts) {
        ferry::set_error("%s: expert id %lld of token %lld is out of range [0, %lld)", who,
                         (long long)e, (long long)t, (long long)experts);
        return -3;
      }
      const bool repeated = seen[(size_t)e] == tt;
      seen[(size_t)e] = tt;
      if (repeated) {
        ferry::set_error("%s: expert id %lld repeated in token %lld", who, (long long)e,
                         (long long)t);
        return -3;
      }
      ++h[e];
    }
  }
  demand->resize((size_t)experts);
  for (int64_t e = 0; e < experts; ++e)
    (*demand)[(size_t)e] = hist[(size_t)e] + hist[(size_t)(experts + e)] +
                           hist[(size_t)(2 * experts + e)] + hist[(size_t)(3 * experts + e)];
  return 0;
}

// The demand of a call whose IDs ferry_history_count checked and counted on the device: the sum
// of its records.  0, or -3 with the error set.
int64_t sum_records(const int32_t* records, int64_t tokens, int64_t experts,
                    std::vector<int64_t>* demand, const char* who) {
  const int64_t blocks = (tokens + ferry::kCountTokens - 1) / ferry::kCountTokens;
  const int64_t words = ferry::count_record_words(experts);
  std::vector<int32_t> sum((size_t)(2 * (words - 1)), 0);
  for (int64_t b = 0; b < blocks; ++b) {
    const int32_t* rec = records + b * words;
    if (rec[0] != 0) {
      ferry::set_error("%s: an expert id of token %lld is out of range [0, %lld) or repeated", who,
                       (long long)(b * ferry::kCountTokens + rec[0] - 1), (long long)experts);
      return -3;
    }
    for (int64_t w = 0; w < words - 1; ++w) {
      const uint32_t pair = (uint32_t)rec[1 + w];
      sum[(size_t)(2 * w)] += (int32_t)(pair & 0xFFFF);
      sum[(size_t)(2 * w + 1)] += (int32_t)(pair >> 16);
    }
  }
  demand->assign(sum.begin(), sum.begin() + experts);
  return 0;
}

// plan_layer on each expert's demand: the misses, slot choices and state updates.
int64_t plan_demand(int64_t event, int64_t layer, const std::vector<int64_t>& demand,
                    const float* gate_scores, int64_t* slots, int64_t cap, int64_t* owner,
                    int64_t* last, float* scores, int64_t experts, int64_t* fetches_out) {
  const int64_t base = layer * experts;
  std::memcpy(scores + base, gate_scores, (size_t)experts * sizeof(float));
  std::vector<uint8_t> active((size_t)experts, 0);
  for (int64_t e = 0; e < experts; ++e) active[(size_t)e] = demand[(size_t)e] > 0;
  std::vector<int64_t> misses;
  misses.reserve((size_t)experts);
  for (int64_t e = 0; e < experts; ++e)
    if (active[(size_t)e] && owner[base + e] < 0) misses.push_back(e);
  int64_t admissible = 0;
  for (int64_t i = 0; i < cap; ++i) {
    const int64_t key = slots[i];
    if (key < 0 || !(key / experts == layer && active[(size_t)(key % experts)])) ++admissible;
  }
  const int64_t m = (int64_t)misses.size();
  if (m > admissible) {
    ferry::set_error("missing experts exceed the total admission capacity (%lld > %lld)",
                     (long long)m, (long long)admissible);
    return -1;
  }
  // Repeated ferry_choose_slot calls, one per miss, pick the slots in one fixed order: a slot
  // that receives a miss then holds an expert this layer needs (never chosen again), and no
  // other slot's key, score or last-use tick changes during the call.  So the misses take the
  // first m admissible slots in that order: the empty slots by index, then the others by
  // (score of the key's own layer, last-use tick, key) -- O(cap + m log cap) instead of O(m cap).
  std::vector<int64_t> order;
  order.reserve((size_t)cap);
  int64_t empties = 0;
  for (int64_t i = 0; i < cap; ++i)
    if (slots[i] < 0) {
      order.push_back(i);
      ++empties;
    }
  if (empties < m) {
    // a key whose score is NaN never compares below the running best, so the scan never
    // picks its slot: such slots are no candidates
    for (int64_t i = 0; i < cap; ++i) {
      const int64_t key = slots[i];
      if (key >= 0 && !(key / experts == layer && active[(size_t)(key % experts)]) &&
          !std::isnan(scores[key]))
        order.push_back(i);
    }
    if ((int64_t)order.size() < m) {
      ferry::set_error("no evictable cache slot for key %lld",
                       (long long)(base + misses[order.size()]));
      return -1;
    }
    auto before = [&](int64_t a, int64_t b) {
      const int64_t ka = slots[a], kb = slots[b];
      const double sa = scores[ka], sb = scores[kb];
      if (sa != sb) return sa < sb;
      if (last[ka] != last[kb]) return last[ka] < last[kb];
      return ka < kb;
    };
    const auto first = order.begin() + empties;
    const auto upto = order.begin() + m;
    std::partial_sort(first, upto, order.end(), before);
  }
  for (int64_t i = 0; i < m; ++i) {
    const int64_t key = base + misses[(size_t)i];
    const int64_t slot = order[(size_t)i];
    const int64_t victim = slots[slot];
    if (victim >= 0) owner[victim] = -1;
    slots[slot] = key;
    owner[key] = 0;
    fetches_out[3 * i + 0] = 0;
    fetches_out[3 * i + 1] = key;
    fetches_out[3 * i + 2] = slot;
  }
  for (int64_t e = 0; e < experts; ++e)
    if (active[(size_t)e]) last[base + e] = event + 1;
  return m;
}

template <typename T>
int64_t plan_core(int64_t event, int64_t layer, const T* ids, int64_t tokens, int64_t topk,
                  const float* gate_scores, int64_t* slots, int64_t cap, int64_t* owner,
                  int64_t* last, float* scores, int64_t experts, int64_t* fetches_out,
                  int64_t* destinations_out, int64_t* demand_out, const char* who) {
  ferry::clear_error();
  if (experts <= 0 || topk <= 0 || tokens < 0 || cap < 0 || layer < 0) {
    ferry::set_error("%s: bad sizes", who);
    return -1;
  }
  std::vector<int64_t> demand;
  const int64_t rc = scan_ids(ids, tokens, topk, experts, &demand, who);
  if (rc != 0) return rc;
  const int64_t m = plan_demand(event, layer, demand, gate_scores, slots, cap, owner, last, scores,
                                experts, fetches_out);
  if (m < 0) return m;
  if (destinations_out)
    for (int64_t i = 0; i < tokens * topk; ++i)
      destinations_out[i] = owner[layer * experts + (int64_t)ids[i]];
  if (demand_out) std::memcpy(demand_out, demand.data(), (size_t)experts * sizeof(int64_t));
  return m;
}

// Queue the copies of a plan's misses on the fetch engine (null: plan only).
int64_t fetch_planned(ferry_h2d* h2d, const int64_t* fetches, int64_t m) {
  if (m <= 0 || !h2d) return m;
  std::vector<int64_t> fs((size_t)m), fk((size_t)m);
  for (int64_t j = 0; j < m; ++j) {
    fk[(size_t)j] = fetches[3 * j + 1];
    fs[(size_t)j] = fetches[3 * j + 2];
  }
  return ferry_h2d_fetch(h2d, fs.data(), fk.data(), m) == 0 ? m : -2;
}

}  // namespace

extern "C" int64_t ferry_plan_layer(int64_t event, int64_t layer, const int64_t* selected,
                                    int64_t tokens, int64_t topk, const float* gate_scores,
                                    int64_t* slots, int64_t cap, int64_t* owner, int64_t* last,
                                    float* scores, int64_t experts, int64_t* fetches_out,
                                    int64_t* destinations_out) {
  return plan_core(event, layer, selected, tokens, topk, gate_scores, slots, cap, owner, last,
                   scores, experts, fetches_out, destinations_out, nullptr, "plan_layer");
}

extern "C" void ferry_layer_slots(const int64_t* slots, int64_t cap, int64_t layer,
                                  int64_t experts, int64_t* lookup) {
  for (int64_t e = 0; e < experts; ++e) lookup[e] = -1;
  for (int64_t i = 0; i < cap; ++i) {
    const int64_t key = slots[i];
    if (key >= 0 && key / experts == layer) lookup[key % experts] = i;
  }
}

extern "C" int ferry_layer_lists(const int64_t* slots, int64_t cap, int64_t layer, int64_t experts,
                                 const int64_t* demand, const int64_t* fetches, int64_t m,
                                 int32_t* slot_of, int32_t* lists, int64_t* list_slots,
                                 int64_t* sizes) {
  ferry::clear_error();
  if (!slots || !demand || !slot_of || !lists || !list_slots || !sizes || (m > 0 && !fetches) ||
      cap < 0 || layer < 0 || experts <= 0 || m < 0) {
    ferry::set_error("layer_lists: bad arguments");
    return 2;
  }
  for (int64_t e = 0; e < experts; ++e) slot_of[e] = -1;
  for (int64_t i = 0; i < cap; ++i) {
    const int64_t key = slots[i];
    if (key >= 0 && key / experts == layer) slot_of[key % experts] = (int32_t)i;
  }
  std::vector<uint8_t> fetched((size_t)experts, 0);
  for (int64_t j = 0; j < m; ++j) {
    const int64_t e = fetches[3 * j + 1] - layer * experts;
    if (e < 0 || e >= experts) {
      ferry::set_error("layer_lists: a fetch of another layer");
      return 2;
    }
    fetched[(size_t)e] = 1;
  }
  // lists: active, resident, fetched experts, each followed by its row counts
  int64_t n[3] = {0, 0, 0}, most[3] = {0, 0, 0}, least[3] = {0, 0, 0};
  for (int64_t e = 0; e < experts; ++e) {
    const int64_t r = demand[e];
    if (r <= 0) continue;
    for (const int l : {0, fetched[(size_t)e] ? 2 : 1}) {
      int32_t* list = lists + 2 * l * experts;
      list[n[l]] = (int32_t)e;
      list[experts + n[l]] = (int32_t)r;
      list_slots[l * experts + n[l]] = slot_of[e];
      most[l] = n[l] == 0 || r > most[l] ? r : most[l];
      least[l] = n[l] == 0 || r < least[l] ? r : least[l];
      ++n[l];
    }
  }
  for (int l = 0; l < 3; ++l) {
    sizes[3 * l] = n[l];
    sizes[3 * l + 1] = most[l];
    sizes[3 * l + 2] = least[l];
  }
  return 0;
}

extern "C" int64_t ferry_plan_fetch(int64_t event, int64_t layer, const uint8_t* ids,
                                    int64_t tokens, int64_t topk, const float* gate_scores,
                                    int64_t* slots, int64_t cap, int64_t* owner, int64_t* last,
                                    float* scores, int64_t experts, int64_t* fetches_out,
                                    int64_t* destinations_out, int64_t* demand_out,
                                    ferry_h2d* h2d) {
  const int64_t m = plan_core(event, layer, ids, tokens, topk, gate_scores, slots, cap, owner,
                              last, scores, experts, fetches_out, destinations_out, demand_out,
                              "plan_fetch");
  return fetch_planned(h2d, fetches_out, m);
}

extern "C" int64_t ferry_plan_fetch_counts(int64_t event, int64_t layer, const int32_t* records,
                                           int64_t tokens, const float* gate_scores,
                                           int64_t* slots, int64_t cap, int64_t* owner,
                                           int64_t* last, float* scores, int64_t experts,
                                           int64_t* fetches_out, int64_t* demand_out,
                                           ferry_h2d* h2d) {
  ferry::clear_error();
  if (experts <= 0 || tokens < 0 || cap < 0 || layer < 0) {
    ferry::set_error("plan_fetch_counts: bad sizes");
    return -1;
  }
  std::vector<int64_t> demand;
  const int64_t rc = sum_records(records, tokens, experts, &demand, "plan_fetch_counts");
  if (rc != 0) return rc;
  const int64_t m = plan_demand(event, layer, demand, gate_scores, slots, cap, owner, last, scores,
                                experts, fetches_out);
  if (m < 0) return m;
  if (demand_out) std::memcpy(demand_out, demand.data(), (size_t)experts * sizeof(int64_t));
  return fetch_planned(h2d, fetches_out, m);
}
