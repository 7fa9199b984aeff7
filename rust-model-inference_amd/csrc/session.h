// What every decoder session has: its device allocations, the token and sampling arrays, stop ids, and the
// generation loop that schedules prompt passes and single steps (Qwen3Session::generate_inner,
// src/models/qwen3.rs:581-1158, is the loop's model).
#pragma once

#include <functional>
#include <vector>

#include "rmi_internal.h"

constexpr uint32_t kArgmaxGroups = 256;
// Workgroups that share a position's logits: all of them for a few positions; for many, sixteen a compute unit in all, so that
// a thread has more to read than its workgroup's reduction takes (128 positions of 151936: 45.8 us with 256 a position, 16.5
// with 32 and four loads a thread under way).
inline uint32_t rmi_argmax_groups(uint32_t positions) {
    const uint32_t n = 4096 / (positions ? positions : 1);
    return n >= kArgmaxGroups ? kArgmaxGroups : n < 1 ? 1 : n;
}
constexpr size_t kTopBytes = 16;  // one Top of device_sample.h

// Called while a pass is enqueued, with a position and where its logits lie at that point of the stream.
using RmiLogitsOf = std::function<void(uint32_t step, const float *logits)>;

struct RmiSession {
    uint32_t vocab = 0, capacity = 0;
    uint32_t *tok = nullptr, *step_argmax = nullptr, *nonfinite = nullptr;
    float *step_top2 = nullptr;
    void *partial = nullptr;
    void *params = nullptr;          // StepParams in HBM
    std::vector<void *> owned;       // every device allocation but the weights', freed with the session
    std::vector<uint32_t> stop_ids;  // generation ends before the first of these (EOS, im_end)
    uint32_t prompt_pass = 0;        // prompt positions per pass, 0 = every position its own step

    RmiSession() = default;
    RmiSession(const RmiSession &) = delete;
    RmiSession &operator=(const RmiSession &) = delete;
    virtual ~RmiSession();

    // a device allocation that lives as long as the session; nullptr and the error text on failure
    void *alloc_bytes(size_t nbytes, bool zero);
    template <typename T>
    T *alloc(size_t count, bool zero = false) {
        return static_cast<T *>(alloc_bytes(count * sizeof(T), zero));
    }
    float *upload(const float *host, size_t n);
    bool alloc_sampling();  // the arrays above, for `capacity` positions

    // A new sequence begins at position 0.
    virtual void begin_sequence() {}
    // One position: its logits in step_logits(), its argmax, top two logits and the next token on the device.
    virtual int enqueue_step(uint32_t step, hipStream_t st) = 0;
    virtual const float *step_logits() const = 0;
    // Whether the prompt positions step0 .. step0 + n - 1 can go through one pass.
    virtual bool pass_possible(uint32_t step0, uint32_t n) const = 0;
    // Such a pass, after which the session stands where a single step would have left it.  want (ascending, below n):
    // the positions whose logits the caller reads, through `of`; a session may compute more.  sample: the pass ends the
    // prompt.
    virtual int enqueue_pass(uint32_t step0, uint32_t n, const uint32_t *want, uint32_t n_want, bool sample, hipStream_t st, const RmiLogitsOf &of) = 0;
    virtual uint32_t max_pass_want() const { return 0xffffffffu; }
    // How many positions from `step` on, up to `most`, one launch can take one after the other; 0: none.
    virtual uint32_t walk_steps(uint32_t step, uint32_t most) const { (void)step, (void)most; return 0; }
    // Such a launch; afterwards the session stands where the last of n single steps would have left it, with the last one's
    // logits in step_logits() if keep_logits.
    virtual int enqueue_walk(uint32_t step, uint32_t n, uint32_t n_prompt, bool keep_logits, hipStream_t st) {
        (void)step, (void)n, (void)n_prompt, (void)keep_logits, (void)st;
        return RMI_HIP_E_INVALID;
    }
    // Whether a walk enqueued before could not finish (asked behind a synchronisation); walk_steps gives 0 from then on.
    virtual bool walk_gave_up() { return false; }
    // The tag behind which the next walk's words begin: 0, or more than any before it.
    virtual void walk_tags_from(uint32_t tag0) { (void)tag0; }
    uint64_t walks_enqueued = 0, walks_given_up = 0;  // launches, and how often walk_gave_up said so
};
// A session's call that keeps the GPU busy is one of these while it lasts; how many there are in the process.
struct RmiSessionBusy {
    RmiSessionBusy();
    ~RmiSessionBusy();
    RmiSessionBusy(const RmiSessionBusy &) = delete;
    RmiSessionBusy &operator=(const RmiSessionBusy &) = delete;
};
uint32_t rmi_sessions_busy();
// for tests: the two counts, and walk_tags_from
void rmi_session_walk_counts(const RmiSession *s, uint64_t counts[2]);
void rmi_session_walk_tags_from(RmiSession *s, uint32_t tag0);

// rmi_hip_<model>_generate: see rmi_hip_qwen3_generate in the header
int rmi_session_generate(RmiSession *s, const uint32_t *prompt, uint32_t n_prompt, uint32_t max_new, uint32_t *generated,
                         uint32_t *step_argmax, float *step_top2, const uint32_t *dump_steps, uint32_t n_dump,
                         float *dump_logits, double *seconds);
int rmi_session_set_stop_ids(RmiSession *s, const uint32_t *ids, uint32_t n_ids);
