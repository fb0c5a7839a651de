# The HIP sources of libgptoss_moe.so, for its own build and the sanitizer's.
SOURCES := moe_route moe_experts moe_decode moe_prefill moe_midstream moe_stages moe_checkpoint moe_stack moe_capi
