// GENERATED by tools/gen_rust_ffi.py from include/nvr.h — do not edit.  Raw declarations of libnvr.so for the reference crate
// (src/ffi.rs there).  Not compiled in the build image (no Rust toolchain); kept in sync with the header by
// tests/test_host_parity.py::test_rust_ffi_is_in_sync_with_the_header.
#![allow(non_camel_case_types, dead_code)]
use std::os::raw::{c_char, c_int, c_void};

#[repr(C)]
pub struct nvr_model_spec_t {
    _private: [u8; 0],
}
#[repr(C)]
pub struct nvr_seq_t {
    _private: [u8; 0],
}
#[repr(C)]
pub struct nvr_block_manager_t {
    _private: [u8; 0],
}
#[repr(C)]
pub struct nvr_scheduler_t {
    _private: [u8; 0],
}
#[repr(C)]
pub struct nvr_model_runner_t {
    _private: [u8; 0],
}
#[repr(C)]
pub struct nvr_local_group_t {
    _private: [u8; 0],
}
#[repr(C)]
pub struct nvr_engine_t {
    _private: [u8; 0],
}

pub const NVR_OK: i32 = 0;
pub const NVR_ERR_NO_FREE_BLOCKS: i32 = -1;
pub const NVR_ERR_ALREADY_ALLOCATED: i32 = -2;
pub const NVR_ERR_NOT_ALLOCATED: i32 = -3;
pub const NVR_ERR_LEN_MISMATCH: i32 = -4;
pub const NVR_ERR_NOTHING_TO_SCHEDULE: i32 = -5;
pub const NVR_ERR_INVARIANT: i32 = -6;
pub const NVR_ERR_INVALID_ARG: i32 = -7;
pub const NVR_ERR_HIP: i32 = -8;
pub const NVR_ERR_RCCL: i32 = -9;
pub const NVR_ERR_UNSUPPORTED: i32 = -10;
pub const NVR_SEQ_WAITING: i32 = 0;
pub const NVR_SEQ_RUNNING: i32 = 1;
pub const NVR_SEQ_FINISHED: i32 = 2;
pub const NVR_SEQ_PREEMPTED: i32 = 3;
pub const NVR_SEQ_ERROR: i32 = 4;
pub const NVR_ACT_SILU: i32 = 0;
pub const NVR_ACT_GELU: i32 = 1;
pub const NVR_ACT_RELU: i32 = 2;
pub const NVR_ACT_SILU_AND_MUL: i32 = 3;
pub const NVR_ACT_GELU_AND_MUL: i32 = 4;
pub const NVR_TOKENIZE_MAX_CHARS: usize = 100;
pub const NVR_LM_HEAD_MAX_PARTS: usize = 2048;

/// `typedef int (*nvr_stream_fn)(const nvr_sequence_output *out, void *user);` (non-zero return = receiver dropped)
pub type nvr_stream_fn = Option<unsafe extern "C" fn(out: *const nvr_sequence_output, user: *mut c_void) -> c_int>;

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_sampling_params {
    pub temperature: f32,
    pub max_tokens: u64,
    pub ignore_eos: i32,
    pub has_top_p: i32,
    pub top_p: f32,
    pub has_top_k: i32,
    pub top_k: u64,
    pub has_repetition_penalty: i32,
    pub repetition_penalty: f32,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_config {
    pub max_num_batched_tokens: u64,
    pub max_num_seqs: u64,
    pub max_model_len: u64,
    pub gpu_memory_utilization: f32,
    pub tensor_parallel_size: u64,
    pub enforce_eager: i32,
    pub has_eos: i32,
    pub eos_token_id: i64,
    pub kvcache_block_size: u64,
    pub num_kvcache_blocks: i64,
    pub tensor_parallel_rank: u64,
    pub device_ordinal: i32,
    pub sample_seed: u64,
    pub skip_block_size_check: i32,
    pub decode_chain: u32,
    pub recompute_cached_prefix: i32,
    pub enable_chunked_prefill: i32,
    pub async_decode: i32,
    pub shared_prefix_min_seqs: i32,
    pub device: [c_char; 16],
    pub dtype: [c_char; 16],
    pub num_state_slots: u64,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_model_config {
    pub vocab_size: u64,
    pub hidden_size: u64,
    pub intermediate_size: u64,
    pub num_hidden_layers: u64,
    pub num_attention_heads: u64,
    pub num_key_value_heads: u64,
    pub head_dim: u64,
    pub max_position_embeddings: u64,
    pub rms_norm_eps: f32,
    pub rope_theta: f64,
    pub tie_word_embeddings: i32,
    pub init_std: f32,
    pub seed: u64,
    pub qk_norm: i32,
    pub use_bias: i32,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_bm_stats {
    pub total_blocks: u64,
    pub free_blocks: u64,
    pub used_blocks: u64,
    pub cached_blocks: u64,
    pub block_size: u64,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_block_info {
    pub block_id: u64,
    pub ref_count: u64,
    pub has_hash: i32,
    pub hash: u64,
    pub num_tokens: u64,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_sched_stats {
    pub total_sequences: u64,
    pub waiting_sequences: u64,
    pub running_sequences: u64,
    pub finished_sequences: u64,
    pub preemptions: u64,
    pub prefill_batches: u64,
    pub decode_batches: u64,
    pub avg_prefill_batch_size: f64,
    pub avg_decode_batch_size: f64,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_step_info {
    pub is_prefill: i32,
    pub num_seqs: u64,
    pub num_tokens: u64,
    pub num_finished: u64,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_engine_stats {
    pub scheduler: nvr_sched_stats,
    pub total_blocks: u64,
    pub free_blocks: u64,
    pub used_blocks: u64,
    pub utilization: f64,
    pub is_running: i32,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_health_status {
    pub is_healthy: i32,
    pub memory_pressure: f64,
    pub active_sequences: u64,
    pub waiting_sequences: u64,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_sequence_output {
    pub seq_id: u64,
    pub text: *const c_char,
    pub text_len: usize,
    pub token_ids: *const i64,
    pub num_tokens: usize,
    pub completion_token_ids: *const i64,
    pub num_prompt_tokens: usize,
    pub num_completion_tokens: usize,
    pub status: i32,
}

#[repr(C)]
#[derive(Clone, Copy)]
pub struct nvr_attn_meta {
    pub is_prefill: i32,
    pub cu_seqlens_q: *const i32,
    pub cu_seqlens_k: *const i32,
    pub max_seqlen_q: i32,
    pub max_seqlen_k: i32,
    pub slot_mapping: *const i32,
    pub context_lens: *const i32,
    pub block_tables: *const i32,
    pub max_blocks: i32,
    pub batch: i32,
    pub max_context_len: i32,
}

#[link(name = "nvr")]
extern "C" {
    pub fn nvr_last_error() -> *const c_char;
    pub fn nvr_last_status() -> c_int;
    pub fn nvr_version() -> *const c_char;
    pub fn nvr_sampling_params_default(sp: *mut nvr_sampling_params);
    pub fn nvr_sampling_params_validate(sp: *const nvr_sampling_params) -> c_int;
    pub fn nvr_config_default(cfg: *mut nvr_config);
    pub fn nvr_config_validate(cfg: *const nvr_config) -> c_int;
    pub fn nvr_model_config_default(mc: *mut nvr_model_config);
    pub fn nvr_model_config_qwen3_0_6b(mc: *mut nvr_model_config);
    pub fn nvr_model_config_qwen3_8b(mc: *mut nvr_model_config);
    pub fn nvr_model_config_validate(mc: *const nvr_model_config, tp: u64) -> c_int;
    pub fn nvr_model_registry_size() -> usize;
    pub fn nvr_model_registry_name(i: usize) -> *const c_char;
    pub fn nvr_model_spec_from_json(config_json_text: *const c_char) -> *mut nvr_model_spec_t;
    pub fn nvr_model_spec_destroy(spec: *mut nvr_model_spec_t);
    pub fn nvr_model_spec_architecture(spec: *const nvr_model_spec_t) -> *const c_char;
    pub fn nvr_model_spec_family(spec: *const nvr_model_spec_t) -> i32;
    pub fn nvr_model_spec_dense(spec: *const nvr_model_spec_t, out: *mut nvr_model_config) -> c_int;
    pub fn nvr_model_spec_vocab(spec: *const nvr_model_spec_t) -> u64;
    pub fn nvr_model_spec_num_layer_runs(spec: *const nvr_model_spec_t) -> u64;
    pub fn nvr_seq_create(prompt: *const i64, n: usize, sp: *const nvr_sampling_params, block_size: usize) -> *mut nvr_seq_t;
    pub fn nvr_seq_destroy(s: *mut nvr_seq_t);
    pub fn nvr_seq_reset_id_counter();
    pub fn nvr_seq_id(s: *const nvr_seq_t) -> u64;
    pub fn nvr_seq_status(s: *const nvr_seq_t) -> i32;
    pub fn nvr_seq_len(s: *const nvr_seq_t) -> usize;
    pub fn nvr_seq_num_prompt_tokens(s: *const nvr_seq_t) -> usize;
    pub fn nvr_seq_num_completion_tokens(s: *const nvr_seq_t) -> usize;
    pub fn nvr_seq_num_cached_tokens(s: *const nvr_seq_t) -> usize;
    pub fn nvr_seq_num_computed_tokens(s: *const nvr_seq_t) -> usize;
    pub fn nvr_seq_chunk(s: *const nvr_seq_t, start: *mut usize, len: *mut usize);
    pub fn nvr_seq_last_token(s: *const nvr_seq_t) -> i64;
    pub fn nvr_seq_num_blocks(s: *const nvr_seq_t) -> usize;
    pub fn nvr_seq_last_block_num_tokens(s: *const nvr_seq_t) -> usize;
    pub fn nvr_seq_token_ids(s: *const nvr_seq_t, ptr: *mut *const i64, len: *mut usize);
    pub fn nvr_seq_block_table(s: *const nvr_seq_t, ptr: *mut *const i32, len: *mut usize);
    pub fn nvr_seq_append_token(s: *mut nvr_seq_t, token: i64);
    pub fn nvr_seq_should_stop(s: *const nvr_seq_t, has_eos: c_int, eos: i64) -> c_int;
    pub fn nvr_seq_preempt(s: *mut nvr_seq_t);
    pub fn nvr_seq_finish(s: *mut nvr_seq_t);
    pub fn nvr_seq_extend(s: *mut nvr_seq_t, tokens: *const i64, n: usize);
    pub fn nvr_seq_set_chunk(s: *mut nvr_seq_t, start: usize, len: usize) -> c_int;
    pub fn nvr_seq_state_slot(s: *const nvr_seq_t) -> i32;
    pub fn nvr_bm_create(num_blocks: usize, block_size: usize) -> *mut nvr_block_manager_t;
    pub fn nvr_bm_destroy(bm: *mut nvr_block_manager_t);
    pub fn nvr_bm_create_stateful(num_blocks: usize, block_size: usize, state_slots: usize) -> *mut nvr_block_manager_t;
    pub fn nvr_bm_can_extend(bm: *const nvr_block_manager_t, s: *const nvr_seq_t) -> c_int;
    pub fn nvr_bm_extend(bm: *mut nvr_block_manager_t, s: *mut nvr_seq_t) -> c_int;
    pub fn nvr_bm_free_state_slots(bm: *const nvr_block_manager_t) -> usize;
    pub fn nvr_bm_compute_hash(tokens: *const i64, n: usize, has_prefix: c_int, prefix: u64) -> u64;
    pub fn nvr_bm_can_allocate(bm: *const nvr_block_manager_t, s: *const nvr_seq_t) -> c_int;
    pub fn nvr_bm_allocate(bm: *mut nvr_block_manager_t, s: *mut nvr_seq_t) -> c_int;
    pub fn nvr_bm_deallocate(bm: *mut nvr_block_manager_t, s: *mut nvr_seq_t) -> c_int;
    pub fn nvr_bm_can_append(bm: *const nvr_block_manager_t, s: *const nvr_seq_t) -> c_int;
    pub fn nvr_bm_may_append(bm: *mut nvr_block_manager_t, s: *mut nvr_seq_t) -> c_int;
    pub fn nvr_bm_get_stats(bm: *const nvr_block_manager_t, out: *mut nvr_bm_stats) -> c_int;
    pub fn nvr_bm_get_block(bm: *const nvr_block_manager_t, block_id: usize, out: *mut nvr_block_info) -> c_int;
    pub fn nvr_bm_free_list(bm: *const nvr_block_manager_t, out: *mut i32, cap: usize) -> usize;
    pub fn nvr_sched_create(cfg: *const nvr_config) -> *mut nvr_scheduler_t;
    pub fn nvr_sched_destroy(sc: *mut nvr_scheduler_t);
    pub fn nvr_sched_add_sequence(sc: *mut nvr_scheduler_t, s: *mut nvr_seq_t) -> c_int;
    pub fn nvr_sched_schedule(sc: *mut nvr_scheduler_t, out: *mut *mut nvr_seq_t, cap: usize, n: *mut usize, is_prefill: *mut c_int) -> c_int;
    pub fn nvr_sched_postprocess(sc: *mut nvr_scheduler_t, seqs: *const *mut nvr_seq_t, token_ids: *const i64, n: usize) -> c_int;
    pub fn nvr_sched_is_finished(sc: *const nvr_scheduler_t) -> c_int;
    pub fn nvr_sched_preempt_all(sc: *mut nvr_scheduler_t);
    pub fn nvr_sched_get_stats(sc: *const nvr_scheduler_t, out: *mut nvr_sched_stats) -> c_int;
    pub fn nvr_sched_get_block_stats(sc: *const nvr_scheduler_t, out: *mut nvr_bm_stats) -> c_int;
    pub fn nvr_sched_queue_lengths(sc: *const nvr_scheduler_t, waiting: *mut usize, running: *mut usize);
    pub fn nvr_sched_memory_pressure(sc: *const nvr_scheduler_t) -> f64;
    pub fn nvr_sched_block_manager(sc: *mut nvr_scheduler_t) -> *mut nvr_block_manager_t;
    pub fn nvr_sched_take_finished(sc: *mut nvr_scheduler_t, out: *mut *mut nvr_seq_t, cap: usize) -> usize;
    pub fn nvr_runner_create(cfg: *const nvr_config, mc: *const nvr_model_config) -> *mut nvr_model_runner_t;
    pub fn nvr_runner_destroy(r: *mut nvr_model_runner_t);
    pub fn nvr_runner_create_spec(cfg: *const nvr_config, spec: *const nvr_model_spec_t) -> *mut nvr_model_runner_t;
    pub fn nvr_runner_execute_step(r: *mut nvr_model_runner_t, seqs: *const *mut nvr_seq_t, n: usize, want_rows: *const i32, n_want: usize, logits_dev: *mut *const f32) -> c_int;
    pub fn nvr_runner_execute_model(r: *mut nvr_model_runner_t, seqs: *const *mut nvr_seq_t, n: usize, is_prefill: c_int, logits_dev: *mut *const f32) -> c_int;
    pub fn nvr_runner_sample_tokens(r: *mut nvr_model_runner_t, seqs: *const *mut nvr_seq_t, n: usize, out_ids: *mut i64) -> c_int;
    pub fn nvr_runner_copy_logits(r: *mut nvr_model_runner_t, host_out: *mut f32, rows: usize) -> c_int;
    pub fn nvr_runner_load_tensor(r: *mut nvr_model_runner_t, name: *const c_char, dtype: c_int, shape: *const i64, ndim: c_int, host_data: *const c_void) -> c_int;
    pub fn nvr_runner_copy_weight(r: *mut nvr_model_runner_t, local_name: *const c_char, host_out: *mut u16, cap_elems: usize, rows: *mut i64, cols: *mut i64) -> c_int;
    pub fn nvr_runner_num_kvcache_blocks(r: *const nvr_model_runner_t) -> u64;
    pub fn nvr_runner_kv_cache(r: *mut nvr_model_runner_t, layer: usize, k_dev: *mut *mut c_void, v_dev: *mut *mut c_void) -> c_int;
    pub fn nvr_runner_stream(r: *mut nvr_model_runner_t) -> *mut c_void;
    pub fn nvr_runner_replay_last_decode_graph(r: *mut nvr_model_runner_t, n: c_int) -> c_int;
    pub fn nvr_comm_unique_id(id_out: *mut u8) -> c_int;
    pub fn nvr_runner_init_comm(r: *mut nvr_model_runner_t, id: *const u8) -> c_int;
    pub fn nvr_runner_comm_selftest(r: *mut nvr_model_runner_t) -> c_int;
    pub fn nvr_local_group_create(nranks: c_int) -> *mut nvr_local_group_t;
    pub fn nvr_local_group_destroy(g: *mut nvr_local_group_t);
    pub fn nvr_runner_init_comm_local(r: *mut nvr_model_runner_t, g: *mut nvr_local_group_t) -> c_int;
    pub fn nvr_local_group_set_p2p(g: *mut nvr_local_group_t, on: c_int) -> c_int;
    pub fn nvr_runner_p2p_export(r: *mut nvr_model_runner_t, handle: *mut u8) -> c_int;
    pub fn nvr_runner_p2p_attach(r: *mut nvr_model_runner_t, handles: *const u8, devices: *const i32) -> c_int;
    pub fn nvr_runner_p2p_disable(r: *mut nvr_model_runner_t) -> c_int;
    pub fn nvr_runner_p2p_active(r: *const nvr_model_runner_t) -> c_int;
    pub fn nvr_runner_p2p_set_fenced(r: *mut nvr_model_runner_t, on: i32) -> c_int;
    pub fn nvr_runner_p2p_fenced(r: *const nvr_model_runner_t) -> c_int;
    pub fn nvr_runner_p2p_reset(r: *mut nvr_model_runner_t) -> c_int;
    pub fn nvr_runner_comm_drop_rccl(r: *mut nvr_model_runner_t) -> c_int;
    pub fn nvr_runner_last_shared_prefix_len(r: *const nvr_model_runner_t) -> i64;
    pub fn nvr_runner_last_prefill_kv_source(r: *const nvr_model_runner_t) -> c_int;
    pub fn nvr_runner_last_shared_prefix_rows(r: *const nvr_model_runner_t) -> i64;
    pub fn nvr_runner_last_decode_ragged(r: *const nvr_model_runner_t) -> i32;
    pub fn nvr_runner_set_tp_prefill_overlap(r: *mut nvr_model_runner_t, on: i32) -> c_int;
    pub fn nvr_runner_last_overlap_chunks(r: *const nvr_model_runner_t) -> i64;
    pub fn nvr_engine_create(cfg: *const nvr_config, mc: *const nvr_model_config) -> *mut nvr_engine_t;
    pub fn nvr_engine_destroy(e: *mut nvr_engine_t);
    pub fn nvr_engine_create_spec(cfg: *const nvr_config, spec: *const nvr_model_spec_t) -> *mut nvr_engine_t;
    pub fn nvr_engine_add_request(e: *mut nvr_engine_t, prompt: *const i64, n: usize, sp: *const nvr_sampling_params, seq_id_out: *mut u64) -> c_int;
    pub fn nvr_engine_step(e: *mut nvr_engine_t, info: *mut nvr_step_info) -> c_int;
    pub fn nvr_engine_is_finished(e: *const nvr_engine_t) -> c_int;
    pub fn nvr_engine_scheduler(e: *mut nvr_engine_t) -> *mut nvr_scheduler_t;
    pub fn nvr_engine_get_stats(e: *mut nvr_engine_t, out: *mut nvr_engine_stats) -> c_int;
    pub fn nvr_engine_health_check(e: *mut nvr_engine_t, out: *mut nvr_health_status) -> c_int;
    pub fn nvr_engine_shutdown(e: *mut nvr_engine_t) -> c_int;
    pub fn nvr_engine_runner(e: *mut nvr_engine_t) -> *mut nvr_model_runner_t;
    pub fn nvr_engine_last_step(e: *const nvr_engine_t, seq_ids: *mut *const u64, tokens: *mut *const i64, n: *mut usize);
    pub fn nvr_engine_take_finished(e: *mut nvr_engine_t, out: *mut *mut nvr_seq_t, cap: usize) -> usize;
    pub fn nvr_engine_abort_last_batch(e: *mut nvr_engine_t) -> c_int;
    pub fn nvr_engine_ahead_declined(e: *const nvr_engine_t) -> u64;
    pub fn nvr_engine_ahead_launched(e: *const nvr_engine_t) -> u64;
    pub fn nvr_engine_host_times(e: *const nvr_engine_t, out3: *mut f64);
    pub fn nvr_engine_last_batch(e: *const nvr_engine_t, out: *mut *mut nvr_seq_t, cap: usize) -> usize;
    pub fn nvr_tokenize(utf8: *const c_char, nbytes: usize, out: *mut i64, cap: usize, n: *mut usize) -> c_int;
    pub fn nvr_detokenize(ids: *const i64, n: usize, out: *mut c_char, cap: usize, nbytes: *mut usize) -> c_int;
    pub fn nvr_engine_add_prompt(e: *mut nvr_engine_t, utf8: *const c_char, nbytes: usize, sp: *const nvr_sampling_params, seq_id_out: *mut u64) -> c_int;
    pub fn nvr_engine_generate(e: *mut nvr_engine_t, prompts: *const *const c_char, nbytes: *const usize, n: usize, sp: *const nvr_sampling_params, outs: *mut *const nvr_sequence_output, nout: *mut usize) -> c_int;
    pub fn nvr_engine_generate_ids(e: *mut nvr_engine_t, prompts: *const *const i64, lens: *const usize, n: usize, sp: *const nvr_sampling_params, outs: *mut *const nvr_sequence_output, nout: *mut usize) -> c_int;
    pub fn nvr_engine_generate_stream(e: *mut nvr_engine_t, prompts: *const *const c_char, nbytes: *const usize, n: usize, sp: *const nvr_sampling_params, fn_: nvr_stream_fn, user: *mut c_void) -> c_int;
    pub fn nvr_device_count(n: *mut c_int) -> c_int;
    pub fn nvr_device_set(ordinal: c_int) -> c_int;
    pub fn nvr_device_name(buf: *mut c_char, cap: usize) -> c_int;
    pub fn nvr_device_mem_info(free_bytes: *mut u64, total_bytes: *mut u64) -> c_int;
    pub fn nvr_device_malloc(ptr: *mut *mut c_void, bytes: usize) -> c_int;
    pub fn nvr_device_free(ptr: *mut c_void) -> c_int;
    pub fn nvr_device_memset(ptr: *mut c_void, value: c_int, bytes: usize) -> c_int;
    pub fn nvr_memcpy_h2d(dst_dev: *mut c_void, src_host: *const c_void, bytes: usize) -> c_int;
    pub fn nvr_memcpy_d2h(dst_host: *mut c_void, src_dev: *const c_void, bytes: usize) -> c_int;
    pub fn nvr_device_synchronize() -> c_int;
    pub fn nvr_stream_create(stream: *mut *mut c_void) -> c_int;
    pub fn nvr_stream_destroy(stream: *mut c_void) -> c_int;
    pub fn nvr_stream_synchronize(stream: *mut c_void) -> c_int;
    pub fn nvr_event_create(ev: *mut *mut c_void) -> c_int;
    pub fn nvr_event_destroy(ev: *mut c_void) -> c_int;
    pub fn nvr_event_record(ev: *mut c_void, stream: *mut c_void) -> c_int;
    pub fn nvr_stream_wait_event(stream: *mut c_void, ev: *mut c_void) -> c_int;
    pub fn nvr_event_elapsed_ms(start: *mut c_void, stop: *mut c_void, ms: *mut f32) -> c_int;
    pub fn nvr_graph_capture_begin(stream: *mut c_void) -> c_int;
    pub fn nvr_graph_capture_end(stream: *mut c_void, graph_exec: *mut *mut c_void) -> c_int;
    pub fn nvr_graph_launch(graph_exec: *mut c_void, stream: *mut c_void) -> c_int;
    pub fn nvr_graph_destroy(graph_exec: *mut c_void) -> c_int;
    pub fn nvr_ops_set_dtype(dtype: *const c_char) -> c_int;
    pub fn nvr_ops_dtype() -> *const c_char;
    pub fn nvr_embedding(ids: *const i64, T: i64, E: *const u16, Hd: i64, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_rmsnorm(x: *const u16, w: *const u16, eps: f32, T: i64, Hd: i64, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_add_rmsnorm(h: *mut u16, y: *const u16, w: *const u16, eps: f32, T: i64, Hd: i64, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_linear(x: *const u16, ldx: i64, W: *const u16, T: i64, K: i64, N: i64, y: *mut c_void, y_is_f32: c_int, stream: *mut c_void) -> c_int;
    pub fn nvr_lm_head(x: *const u16, ldx: i64, W: *const u16, T: i64, K: i64, N: i64, logits: *mut f32, part_val: *mut f32, part_idx: *mut i32, nparts: *mut i32, stream: *mut c_void) -> c_int;
    pub fn nvr_argmax_partials(part_val: *const f32, part_idx: *const i32, nparts: i32, T: i64, out_idx: *mut i64, out_val: *mut f32, idx_offset: i64, stream: *mut c_void) -> c_int;
    pub fn nvr_linear_splitk(x: *const u16, ldx: i64, W: *const u16, T: i64, K: i64, N: i64, S: i64, slabs: *mut f32, stream: *mut c_void) -> c_int;
    pub fn nvr_add_rmsnorm_slabs(h: *mut u16, slabs: *const f32, S: i64, w: *const u16, eps: f32, T: i64, Hd: i64, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_retile_weight(src: *const u16, dst: *mut u16, N: i64, K: i64, mode: c_int, H: i64, KVH: i64, D: i64, stream: *mut c_void) -> c_int;
    pub fn nvr_linear_tiled(x: *const u16, ldx: i64, W: *const u16, Wt: *const u16, T: i64, K: i64, N: i64, y: *mut c_void, y_is_f32: c_int, stream: *mut c_void) -> c_int;
    pub fn nvr_linear_splitk_tiled(x: *const u16, ldx: i64, W: *const u16, Wt: *const u16, T: i64, K: i64, N: i64, S: i64, slabs: *mut f32, stream: *mut c_void) -> c_int;
    pub fn nvr_linear_silu_mul_tiled(x: *const u16, ldx: i64, W: *const u16, Wt: *const u16, T: i64, K: i64, I: i64, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_linear_qkv_rope_store_tiled(x: *const u16, ldx: i64, W: *const u16, Wt: *const u16, T: i64, K: i64, H: i64, KVH: i64, D: i64, positions: *const i64, slot_mapping: *const i32, cos_t: *const f32, sin_t: *const f32, qkv: *mut u16, k_cache: *mut u16, v_cache: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_lm_head_tiled(x: *const u16, ldx: i64, W: *const u16, Wt: *const u16, T: i64, K: i64, N: i64, logits: *mut f32, part_val: *mut f32, part_idx: *mut i32, nparts: *mut i32, stream: *mut c_void) -> c_int;
    pub fn nvr_decode_splitk_slices(T: i64, K: i64, N: i64) -> c_int;
    pub fn nvr_linear_add_residual(x: *const u16, ldx: i64, W: *const u16, T: i64, K: i64, N: i64, h: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_linear_silu_mul(x: *const u16, ldx: i64, W: *const u16, T: i64, K: i64, I: i64, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_linear_qkv_rope_store(x: *const u16, ldx: i64, W: *const u16, T: i64, K: i64, H: i64, KVH: i64, D: i64, positions: *const i64, slot_mapping: *const i32, cos_t: *const f32, sin_t: *const f32, qkv: *mut u16, k_cache: *mut u16, v_cache: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_rope_store_kv(qkv: *mut u16, positions: *const i64, slot_mapping: *const i32, T: i64, H: i64, KVH: i64, D: i64, cos_t: *const f32, sin_t: *const f32, k_cache: *mut u16, v_cache: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_qk_norm_rope_store_kv(qkv: *mut u16, positions: *const i64, slot_mapping: *const i32, T: i64, H: i64, KVH: i64, D: i64, cos_t: *const f32, sin_t: *const f32, q_norm_w: *const u16, k_norm_w: *const u16, eps: f32, k_cache: *mut u16, v_cache: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_linear_qkv_norm_rope_store(x: *const u16, ldx: i64, W: *const u16, Wt: *const u16, T: i64, K: i64, H: i64, KVH: i64, D: i64, positions: *const i64, slot_mapping: *const i32, cos_t: *const f32, sin_t: *const f32, q_norm_w: *const u16, k_norm_w: *const u16, eps: f32, qkv: *mut u16, k_cache: *mut u16, v_cache: *mut u16, kv_cache_only: c_int, stream: *mut c_void) -> c_int;
    pub fn nvr_rope_table(D: i64, max_pos: i64, theta: f64, cos_dev: *mut f32, sin_dev: *mut f32) -> c_int;
    pub fn nvr_paged_attn_workspace_bytes(B: i64, H: i64, D: i64, max_context_len: i64) -> usize;
    pub fn nvr_paged_attn_decode(q: *const u16, ldq: i64, k_cache: *const u16, v_cache: *const u16, meta: *const nvr_attn_meta, H: i64, KVH: i64, D: i64, block_size: i64, scale: f32, out: *mut u16, workspace: *mut c_void, stream: *mut c_void) -> c_int;
    pub fn nvr_paged_attn_decode_fused(q: *const u16, ldq: i64, k_cache: *const u16, v_cache: *const u16, meta: *const nvr_attn_meta, H: i64, KVH: i64, D: i64, block_size: i64, scale: f32, out: *mut u16, workspace: *mut c_void, tickets: *mut u32, stream: *mut c_void) -> c_int;
    pub fn nvr_paged_attn_decode_shared(q: *const u16, ldq: i64, k_cache: *const u16, v_cache: *const u16, meta: *const nvr_attn_meta, H: i64, KVH: i64, D: i64, block_size: i64, scale: f32, shared_len: i64, rows: *const i32, kv0: *const i32, count: *const i32, out: *mut u16, workspace: *mut c_void, stream: *mut c_void) -> c_int;
    pub fn nvr_attn_prefill_varlen(q: *const u16, k: *const u16, v: *const u16, ld: i64, meta: *const nvr_attn_meta, T: i64, H: i64, KVH: i64, D: i64, scale: f32, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_attn_prefill_paged(q: *const u16, ldq: i64, k_cache: *const u16, v_cache: *const u16, meta: *const nvr_attn_meta, T: i64, H: i64, KVH: i64, D: i64, block_size: i64, scale: f32, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_silu_and_mul(x: *const u16, T: i64, I: i64, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_activation_type_from_str(name: *const c_char, type_out: *mut i32) -> c_int;
    pub fn nvr_activation(type_: i32, x: *const u16, T: i64, cols: i64, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_add_bias(y: *mut u16, b: *const u16, T: i64, N: i64, stream: *mut c_void) -> c_int;
    pub fn nvr_select_last_tokens(h: *const u16, cu_seqlens_q: *const i32, B: i64, Hd: i64, out: *mut u16, stream: *mut c_void) -> c_int;
    pub fn nvr_argmax(logits: *const f32, B: i64, V: i64, out_ids: *mut i64, stream: *mut c_void) -> c_int;
    pub fn nvr_sample_workspace_bytes(B: i64, V: i64) -> usize;
    pub fn nvr_sample(logits: *const f32, B: i64, V: i64, temperature: *const f32, top_k: *const i64, top_p: *const f32, keys: *const u64, out_ids: *mut i64, workspace: *mut c_void, stream: *mut c_void) -> c_int;
    pub fn nvr_sample_key(seed: u64, seq_id: u64, step: u64) -> u64;
    pub fn nvr_weight_key(seed: u64, tensor_id: u64) -> u64;
    pub fn nvr_weight_scale(std: f64) -> f32;
    pub fn nvr_fill_weight(dst: *mut u16, rows: i64, cols: i64, ld: i64, global_cols: i64, row0: i64, col0: i64, key: u64, scale: f32, stream: *mut c_void) -> c_int;
    pub fn nvr_fill_const(dst: *mut u16, n: i64, value: f32, stream: *mut c_void) -> c_int;
}
