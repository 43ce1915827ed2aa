// The gfx950 code objects built from kernels.hip, ingest.hip and prompt.hip,
// linked into the library as read-only data and loaded with hipModuleLoadData at init.
    .section .rodata
    .balign 4096
    .global sml_code_object
    .type sml_code_object, @object
sml_code_object:
    .incbin "kernels.hsaco"
    .global sml_code_object_end
sml_code_object_end:
    .byte 0
    .balign 4096
    .global sml_ingest_object
    .type sml_ingest_object, @object
sml_ingest_object:
    .incbin "ingest.hsaco"
    .global sml_ingest_object_end
sml_ingest_object_end:
    .byte 0
    .balign 4096
    .global sml_prompt_object
    .type sml_prompt_object, @object
sml_prompt_object:
    .incbin "prompt.hsaco"
    .global sml_prompt_object_end
sml_prompt_object_end:
    .byte 0
    .section .note.GNU-stack,"",@progbits
