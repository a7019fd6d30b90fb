// tsa_valid.h -- is an uploaded chain a binary tree?  Plain C++, also compiled by the CPU tests.
#pragma once
#include <stdint.h>
#include <string.h>
#include <vector>

// Every chain must be a binary tree over all 2m-1 nodes rooted at 2m-2 (ids < 2m-1, each node reached
// once); the kernels index label sets with these ids.  Reference check: csrc/treesa_gpu.cu:1127-1145.
struct TsaTreeCheck {
  std::vector<unsigned char> seen = std::vector<unsigned char>(1 << 16);  // by node id: any 16-bit word is an index
  std::vector<int> st;

  bool operator()(const uint32_t* ch, int m) { return ordered(ch, m) || reached(ch, m); }

  // A tree whose children all have smaller ids than their parent, as every start tree's do: the ids fall along any
  // path, so there is no cycle, and the 2m-2 child references name each of the 2m-2 nodes below the root once if none
  // is missing.  One pass without a stack, where the traversal's every push and pop waits for the one before; an annealed
  // tree, whose order is another, leaves it after a few nodes for the traversal.  1024 trees of sat100 uploaded and
  // evaluated: 1121 -> 487 us.
  bool ordered(const uint32_t* ch, int m) {
    const int n = 2 * m - 1;
    unsigned char* const s = seen.data();
    memset(s, 0, (size_t)n);
    for (int i = 0; i < m - 1; i++) {
      const unsigned l = ch[i] & 0xFFFFu, r = ch[i] >> 16, v = (unsigned)(m + i);
      if ((l > r ? l : r) >= v) return false;
      s[l] = 1;
      s[r] = 1;
    }
    unsigned all = 1;
    for (int k = 0; k < n - 1; k++) all &= s[k];
    return all != 0;
  }

  // Any tree: from the root down, every node once.
  bool reached(const uint32_t* ch, int m) {
    const int n = 2 * m - 1;
    memset(seen.data(), 0, (size_t)n);
    st.clear();
    st.push_back(n - 1);
    int cnt = 0;
    while (!st.empty()) {
      const int v = st.back();
      st.pop_back();
      if (v < 0 || v >= n || seen[(size_t)v]) return false;
      seen[(size_t)v] = 1;
      cnt++;
      if (v >= m) {
        st.push_back((int)(ch[v - m] >> 16));
        st.push_back((int)(ch[v - m] & 0xFFFFu));
      }
    }
    return cnt == n;
  }
};
