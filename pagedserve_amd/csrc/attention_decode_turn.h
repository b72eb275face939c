// The body of the loop over keys in attention_decode_block.h: the keys base .. base + KEYS_PER_WAVE of a wave into its
// running maximum, sum and values.  FIRST: `ahead` runs behind the loads.  It is text that stands inside the loop and not a
// lambda or a function of its own: as one of those, inlined, its addresses took twice as many multiplications and decode
// attention 1 to 3 % longer (one request of 12 heads of 64 over 144 keys 5.76 us, this way 5.61).  Only the loop whose first
// turn stands apart has it as a lambda, which is the faster there (with the projection, over 60 keys 4.22 us, as text 4.37).
    Raw8<T> kr[AD_UNROLL], vr[AD_UNROLL];
    bool valid[AD_UNROLL];
    // Every load is unconditional from a clamped address and masked afterwards, so that the
    // table entries, then all keys and values of the iteration, travel together.
    int page[AD_UNROLL], within[AD_UNROLL];
#pragma unroll
    for (int u = 0; u < AD_UNROLL; ++u) {
      const int key = base + u * GROUPS + group;
      const int safe_key = key < range_end ? key : range_end - 1;
      const int logical = page_shift >= 0 ? (safe_key >> page_shift) : safe_key / page_size;
      within[u] = safe_key - logical * page_size;
      const int entry = logical < table_width ? logical : table_width - 1;
      if (prefetched) {
        const int low = __shfl(held0, entry & 63, 64);
        page[u] = low;
        if (table_width > 64) {
          const int high = __shfl(held1, entry & 63, 64);
          page[u] = entry < 64 ? low : high;
        }
      } else {
        page[u] = table[entry];
      }
      valid[u] = key < range_end && logical < table_width;
    }
#pragma unroll
    for (int u = 0; u < AD_UNROLL; ++u) {
      valid[u] = valid[u] && page[u] >= 0 && page[u] < num_pages;
      const int safe_page = valid[u] ? page[u] : 0;
      const int64_t offset =
          (((int64_t)safe_page * kv_heads + kv_head) * page_size + within[u]) * head_dim +
          (has_dims ? dim0 : 0);
      kr[u].template load<NT>(k_pool + offset);
      vr[u].template load<NT>(v_pool + offset);
    }
    if constexpr (FIRST) {
      __builtin_amdgcn_sched_barrier(0);
      ahead();
      __builtin_amdgcn_sched_barrier(0);
    }
    float s[AD_UNROLL];
    float m_new = m;
#pragma unroll
    for (int u = 0; u < AD_UNROLL; ++u) {
      float kf[8];
      kr[u].widen(kf);
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) dot = fmaf(qf[i], kf[i], dot);
      if (!has_dims) dot = 0.f;
      if (LPK <= 16) {
        dot = lanes_sum<(LPK <= 16 ? LPK : 16)>(dot);
      } else {
        dot = lanes_sum<16>(dot);
        dot += __shfl_xor(dot, 16, 64);
      }
      float score = dot * scale_log2;
      // (the cap in the scores' units of log 2)
      if (extra.softcap > 0.f) score = capped_score_as<T>(score, extra.softcap * 1.4426950408889634f);
      s[u] = valid[u] ? score : -INFINITY;
      m_new = fmaxf(m_new, s[u]);
    }
    if (logistic) {
#pragma unroll
      for (int u = 0; u < AD_UNROLL; ++u) {
        const float p = valid[u] ? logistic_weight_as<T>(s[u] + shift) : 0.f;
        float vf[8];
        vr[u].widen(vf);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = valid[u] ? fmaf(p, vf[i], acc[i]) : acc[i];
      }
    } else if (m_new != -INFINITY) {
      const float correction = (m == -INFINITY) ? 0.f : exp2_fast<T>(m - m_new);
      l *= correction;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] *= correction;
#pragma unroll
      for (int u = 0; u < AD_UNROLL; ++u) {
        const float p = valid[u] ? exp2_fast<T>(s[u] - m_new) : 0.f;
        l += p;
        float vf[8];
        vr[u].widen(vf);
        // a masked key was loaded from a clamped address and may hold anything, also NaN
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = valid[u] ? fmaf(p, vf[i], acc[i]) : acc[i];
      }
      m = m_new;
    }
