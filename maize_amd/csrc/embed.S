/* Embeds the gfx950 code objects into libmaize_hip.so. */
    .section .rodata
    .balign 4096
    .global maize_embedded_hsaco
    .type maize_embedded_hsaco, @object
maize_embedded_hsaco:
    .incbin MAIZE_HSACO_PATH
    .global maize_embedded_hsaco_end
    .type maize_embedded_hsaco_end, @object
maize_embedded_hsaco_end:
    .byte 0
    .size maize_embedded_hsaco, maize_embedded_hsaco_end - maize_embedded_hsaco
    .balign 4096
    .global maize_embedded_forms
    .type maize_embedded_forms, @object
maize_embedded_forms:
    .incbin MAIZE_FORMS_PATH
    .byte 0
    .size maize_embedded_forms, . - maize_embedded_forms

    .section .note.GNU-stack,"",@progbits
