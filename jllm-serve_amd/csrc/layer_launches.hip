// The launches of one layer, repeated for the layers that are like it.
//
// A prompt's layers ask the host for six launches each, and through Python each costs 14 us: checks, plans, scratch, the argument
// conversion, the launch. Layers of one kind, size and type ask for the same launches in the same order, with other addresses
// (weights, caches, and the two sets of buffers that take turns between a layer and the next). So Python runs one layer, keeps the calls
// it made, and they are made here for the others: 2.5 to 3 us each.
#include <string.h>

#include <utility>

#include "common.h"
#include "layer_launches.h"

template <typename T>
static T from_word(unsigned long long w) {
  T v;
  if constexpr (sizeof(T) == 8) {
    memcpy(&v, &w, 8);
  } else {  // an int or a float: the word's low half
    static_assert(sizeof(T) == 4, "arguments are pointers, ints and floats");
    const unsigned low = (unsigned)w;
    memcpy(&v, &low, 4);
  }
  return v;
}
template <typename... A, size_t... I>
static int call_with(int (*fn)(A...), const unsigned long long* words, std::index_sequence<I...>) {
  return fn(from_word<A>(words[I])...);
}
template <typename... A>
static int call(int (*fn)(A...), const unsigned long long* words) {
  return call_with(fn, words, std::index_sequence_for<A...>{});
}
template <typename... A>
static constexpr int arity(int (*)(A...)) {
  return (int)sizeof...(A);
}
struct LayerEntry {
  const char* name;
  int args;
  int (*call)(const unsigned long long*);
};
#define ENTRY(fn) {#fn, arity(fn), [](const unsigned long long* words) { return call(fn, words); }},
static const LayerEntry entries[] = {JLLM_LAYER_ENTRIES(ENTRY)};
#undef ENTRY
static constexpr int n_entries = (int)(sizeof(entries) / sizeof(entries[0]));

// The number by which an entry point is named below, or -1: not one of them, or not one of `args` arguments.
extern "C" int jllm_layer_entry(const char* name, int args) {
  for (int i = 0; i < n_entries; ++i)
    if (strcmp(entries[i].name, name) == 0) return entries[i].args == args ? i : -1;
  return -1;
}

// `words`: the calls of a layer, each the entry point's number, the count of its arguments and those, a word each (an int or a float
// in the low half). The words numbered `places` [n_places] become `values`, then the calls are made in order. Returns 0, or -1 with the
// message of the call that failed; one that declines what it took for the layer before is an error too, since those in front of it are made.
extern "C" int jllm_layer_launches(unsigned long long* words, long long n_words, const long long* places, int n_places,
                                   const unsigned long long* values) {
  for (int p = 0; p < n_places; ++p)
    if (places[p] < 2 || places[p] >= n_words) JLLM_FAIL("layer launches: place %lld of %lld words", places[p], n_words);
  int p = 0;  // (places ascend, as they were found)
  for (long long at = 0; at < n_words; at += 2 + (long long)words[at + 1]) {
    if (at + 2 > n_words || words[at] >= (unsigned long long)n_entries || words[at + 1] != (unsigned long long)entries[words[at]].args ||
        at + 2 + (long long)words[at + 1] > n_words)
      JLLM_FAIL("layer launches: no call at word %lld of %lld", at, n_words);
    for (; p < n_places && places[p] < at + 2 + (long long)words[at + 1]; ++p) {
      if (places[p] < at + 2) JLLM_FAIL("layer launches: word %lld names a call", places[p]);
      words[places[p]] = values[p];
    }
    const LayerEntry& e = entries[words[at]];
    const int rc = e.call(words + at + 2);
    if (rc < 0) return -1;
    if (rc > 0) JLLM_FAIL("%s declines for a later layer what it took for the first", e.name);
  }
  return 0;
}
